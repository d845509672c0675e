"""The W8A8 GEMM's smaller tiles (xgen_amd/csrc/gemm_tile.h), one ragged shape per tile (M, N and K no
multiples of the tile or of a 128-byte K step) and one whose K steps are fewer than the tile's slots
where a call takes the tile so: accumulators of sampled rows bit for bit (INT8
against the exact sum, FP8 against the MFMA model; the exact kind within the float32 summation
bound), and the outputs equal, bit for bit, to the same rows of a call with many more rows, which
runs on another tile: an output's products are summed in the same order whatever the tile.  Both calls'
tiles are asked of the library."""
import pytest
import torch

import oracle.ref as R
import xgen_amd  # noqa: F401
from conftest import gemm_tile
from xgen_amd import _native as N

pytestmark = pytest.mark.gpu
xops = torch.ops.xgen_amd
FP32_SUM_REL = 2.0 ** -24

# (M, N, K), the tile it runs on, epilogue options
CASES = [
    ((1, 48, 880), "32x64", torch.bfloat16, torch.bfloat16, N.ACT_NONE),
    ((5, 18256, 848), "32x128", torch.float32, torch.float16, N.ACT_NONE),
    ((33, 8224, 144), "64x64", torch.float16, torch.bfloat16, N.ACT_GELU_TANH),
    ((33, 16752, 1232), "64x128", None, torch.float16, N.ACT_GELU_TANH),
    ((515, 5792, 400), "128x128", torch.bfloat16, torch.bfloat16, N.ACT_GELU_TANH),
    ((1290, 3152, 656), "128x192", torch.float32, torch.bfloat16, N.ACT_NONE),
    ((1411, 5088, 272), "256x128", torch.bfloat16, torch.float16, N.ACT_NONE),
    ((3265, 2448, 1808), "256x192", torch.bfloat16, torch.bfloat16, N.ACT_NONE),
    ((131, 6160, 48), "32x128", None, torch.bfloat16, N.ACT_NONE),
    ((33, 8224, 656), "64x64", torch.float32, torch.float16, N.ACT_NONE),
    ((33, 16752, 48), "64x128", torch.bfloat16, torch.bfloat16, N.ACT_NONE),
    ((333, 9232, 48), "128x128", torch.float16, torch.float16, N.ACT_NONE),
]
# the exact kind's cheapest tile for 33 rows of two K steps is another
OTHER_TILE = {((33, 8224, 144), "fp8_exact"): "32x128"}


IDS = [f"{c[1]}-K{c[0][2]}" for c in CASES]


def name(tile):
    return f"{tile[0]}x{tile[1]}"


def operands(M, Nf, K, kind, dev):
    g = torch.Generator(device=dev).manual_seed(M + Nf + K)
    dt = torch.int8 if kind == "int8" else torch.float8_e4m3fn
    qa, sa = xops.quantize_rows(torch.randn((M, K), generator=g, device=dev).to(torch.bfloat16), dt)
    qw, sw = xops.quantize_rows((torch.randn((Nf, K), generator=g, device=dev) * 0.02).to(torch.bfloat16), dt)
    return qa, sa, qw, sw, (torch.randn((Nf,), generator=g, device=dev) * 0.01), g


def more_rows(t, rows):
    """t's rows, then t's rows again up to `rows` of them."""
    reps = -(-rows // t.shape[0])
    return torch.cat([t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t] * reps)[:rows].view(t.dtype)


@pytest.mark.parametrize("kind", ["fp8", "fp8_exact", "int8"])
@pytest.mark.parametrize("shape,tile,bias_dtype,out_dtype,act", CASES, ids=IDS)
def test_tile(cuda, kind, shape, tile, bias_dtype, out_dtype, act):
    M, Nf, K = shape
    exact_kind = kind == "fp8_exact"
    tile = OTHER_TILE.get((shape, kind), tile)
    assert {name(gemm_tile(kind, M, Nf, K, accumulators=a)) for a in (False, True)} == {tile}
    qa, sa, qw, sw, b, _ = operands(M, Nf, K, kind, cuda)
    bias = None if bias_dtype is None else b.to(bias_dtype)
    out, acc = xops.scaled_mm(qa, qw, sa, sw, bias, out_dtype, act, True, exact_kind)
    plain, _ = xops.scaled_mm(qa, qw, sa, sw, bias, out_dtype, act, False, exact_kind)
    assert torch.equal(out, plain)
    rows = torch.unique(torch.cat([torch.tensor([0, M - 1]), torch.arange(max(0, M - 8), M),
                                   torch.randperm(M, generator=torch.Generator().manual_seed(1))[:24]]))
    a, got = qa.view(torch.uint8)[rows.to(cuda)].view(qa.dtype).cpu(), acc[rows.to(cuda)].cpu()
    if kind == "int8":
        assert torch.equal(got.long(), R.int8_accumulate_exact(a, qw.cpu()))
    elif kind == "fp8":
        assert torch.equal(got, R.fp8_mfma_accumulate(a, qw.cpu()))
    else:
        mag = R.decode_fp8(a).abs() @ R.decode_fp8(qw.cpu()).abs().T
        assert ((got.double() - R.fp8_accumulate_exact(a, qw.cpu())).abs() <= K * FP32_SUM_REL * mag).all()
    big = 4 * M + 12288
    assert name(gemm_tile(kind, big, Nf, K, accumulators=True)) != tile
    wide, wide_acc = xops.scaled_mm(more_rows(qa, big), qw, more_rows(sa, big), sw, bias, out_dtype, act, True, exact_kind)
    assert torch.equal(wide[:M], out) and torch.equal(wide_acc[:M], acc)


@pytest.mark.parametrize("kind", ["fp8", "int8"])
@pytest.mark.parametrize("shape,tile", [c[:2] for c in CASES], ids=IDS)
def test_tile_gated_residual(cuda, kind, shape, tile):
    """The gated epilogue equals the plain one followed by the gated residual op, bit for bit, indices
    outside the table (NaN rows) included."""
    M, Nf, K = shape
    assert name(gemm_tile(kind, M, Nf, K, gated=True)) == tile
    qa, sa, qw, sw, b, g = operands(M, Nf, K, kind, cuda)
    bias = b.to(torch.bfloat16)
    residual = torch.randn((M, Nf), generator=g, device=cuda).to(torch.bfloat16)
    gate = torch.randn((7, Nf), generator=g, device=cuda).to(torch.bfloat16)
    seq = M // 3 if M % 3 == 0 else M
    indices = torch.randint(0, 7, (seq,), generator=g, device=cuda)
    indices[seq // 2] = 7 if seq > 1 else indices[0]
    indices[seq - 1] = -1 if seq > 2 else indices[0]
    out = xops.scaled_mm_gate_residual(qa, qw, sa, sw, bias, residual, gate, indices)
    plain, _ = xops.scaled_mm(qa, qw, sa, sw, bias, torch.bfloat16, N.ACT_NONE, False)
    want = xops.gate_residual(residual.reshape(-1, seq, Nf), plain.reshape(-1, seq, Nf), gate, indices).reshape(M, Nf)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
