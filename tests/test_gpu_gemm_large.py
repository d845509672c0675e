"""The W8A8 GEMM's 256 x 256 kernel (xgen_amd/csrc/gemm_w8a8.hip) on ragged calls of more tiles than it has
workgroups: M, N and K no multiples of a tile or a K step, every epilogue, strided operands, the gated
residual with token positions that repeat and indices outside the table.  The tile of each call, and of the
call it is compared with, is asked of the library."""
import pytest
import torch

import oracle.ref as R
import xgen_amd  # noqa: F401
from conftest import gemm_tile
from test_gpu_gemm_tiles import FP32_SUM_REL, operands
from xgen_amd import _native as N

pytestmark = pytest.mark.gpu
xops = torch.ops.xgen_amd
LARGE = (256, 256)

# 17 to 33 x 37 tiles: two to five per workgroup; one, two or three and nine K steps
SHAPES = [(4109, 9232, 80), (4109, 9232, 272), (8197, 9232, 1104)]


def sampled_rows(M, dev):
    """The first and last row of the first, a middle and the last, partial tile-row, and 16 others."""
    tiles = [0, M // 256 // 2 * 256, M // 256 * 256]
    edges = [r for t in tiles for r in (t, min(t + 255, M - 1))]
    others = torch.randperm(M, generator=torch.Generator().manual_seed(1))[:16]
    return torch.unique(torch.cat([torch.tensor(edges), others])).to(dev)


def take(t, rows):
    return t.view(torch.uint8)[rows].view(t.dtype) if t.dtype == torch.float8_e4m3fn else t[rows]


def embed(t, cols, first):
    big = torch.zeros((t.shape[0], cols), dtype=t.dtype, device=t.device)
    big[:, first:first + t.shape[1]] = t
    return big[:, first:first + t.shape[1]]


def check_accumulators(kind, acc, a, w):
    a, w, acc = a.cpu(), w.cpu(), acc.cpu()
    if kind == "int8":
        assert torch.equal(acc.long(), R.int8_accumulate_exact(a, w))
    elif kind == "fp8":
        assert torch.equal(acc, R.fp8_mfma_accumulate(a, w))
    else:
        bound = a.shape[1] * FP32_SUM_REL * (R.decode_fp8(a).abs() @ R.decode_fp8(w).abs().T)
        assert ((acc.double() - R.fp8_accumulate_exact(a, w)).abs() <= bound).all()


@pytest.mark.parametrize("kind", ["fp8", "fp8_exact", "int8"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_accumulators(cuda, kind, shape):
    """Accumulators of sampled rows, all columns: INT8 against the exact sum, FP8 against the MFMA model, the
    exact kind within the float32 summation bound."""
    M, Nf, K = shape
    exact = kind == "fp8_exact"
    assert gemm_tile(kind, M, Nf, K, accumulators=True) == gemm_tile(kind, M, Nf, K) == LARGE
    qa, sa, qw, sw, b, _ = operands(M, Nf, K, kind, cuda)
    out, acc = xops.scaled_mm(qa, qw, sa, sw, b, torch.bfloat16, N.ACT_NONE, True, exact)
    plain, _ = xops.scaled_mm(qa, qw, sa, sw, b, torch.bfloat16, N.ACT_NONE, False, exact)
    assert torch.equal(out.view(torch.int16), plain.view(torch.int16))
    rows = sampled_rows(M, cuda)
    check_accumulators(kind, acc[rows], take(qa, rows), qw)


@pytest.mark.parametrize("kind", ["fp8", "fp8_exact", "int8"])
def test_long_k_accumulators(cuda, kind):
    """K = 12,304 (97 K steps, the last of 16 bytes): accumulators of sampled rows and columns."""
    M, Nf, K = 8205, 12304, 12304
    assert gemm_tile(kind, M, Nf, K, accumulators=True) == LARGE
    qa, sa, qw, sw, _, _ = operands(M, Nf, K, kind, cuda)
    _, acc = xops.scaled_mm(qa, qw, sa, sw, None, torch.bfloat16, N.ACT_NONE, True, kind == "fp8_exact")
    rows = sampled_rows(M, cuda)
    cols = torch.unique(torch.tensor([0, 255, 256, 12287, 12288, 12303, *range(5000, 5032)])).to(cuda)
    check_accumulators(kind, acc[rows][:, cols], take(qa, rows), take(qw, cols))


@pytest.mark.parametrize("kind", ["fp8", "fp8_exact", "int8"])
@pytest.mark.parametrize("act", [N.ACT_NONE, N.ACT_GELU_TANH])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16])
def test_epilogue(cuda, kind, act, out_dtype):
    """Every bias dtype and none, scales per token or tensor against per channel or tensor, both output dtypes,
    with and without GELU: sampled rows bit for bit those of a call on these rows alone, which runs on a
    smaller tile (whose epilogue the oracle checks), strided operands among them."""
    M, Nf, K = SHAPES[1]
    exact = kind == "fp8_exact"
    qa, sa, qw, sw, b, _ = operands(M, Nf, K, kind, cuda)
    rows = sampled_rows(M, cuda)
    assert gemm_tile(kind, M, Nf, K) == LARGE != gemm_tile(kind, len(rows), Nf, K)
    few = take(qa, rows)
    strided = embed(qa, K + 48, 16), embed(qw, K + 64, 32)
    assert strided[0].stride(0) == K + 48 and strided[0].data_ptr() % 16 == 0
    for bias in (None, b, b.to(torch.bfloat16), b.to(torch.float16)):
        for sa_, sw_ in ((sa, sw), (sa[:1].clone(), sw[:1].clone()), (sa, sw[:1].clone()), (sa[:1].clone(), sw)):
            want, _ = xops.scaled_mm(few, qw, sa_[rows] if sa_.numel() > 1 else sa_, sw_, bias, out_dtype, act, False, exact)
            for x, w in ((qa, qw), strided):
                out, _ = xops.scaled_mm(x, w, sa_, sw_, bias, out_dtype, act, False, exact)
                assert torch.equal(out[rows].view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("kind", ["fp8", "int8"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_gated_residual(cuda, kind, shape):
    """seq below M, indices outside the table (NaN rows), contiguous and strided residual, gate and operand rows:
    the plain product followed by the gated residual op, bit for bit."""
    M, Nf, K = shape
    assert gemm_tile(kind, M, Nf, K, gated=True) == gemm_tile(kind, M, Nf, K) == LARGE
    qa, sa, qw, sw, b, g = operands(M, Nf, K, kind, cuda)
    bias = b.to(torch.bfloat16)
    residual = torch.randn((M, Nf), generator=g, device=cuda).to(torch.bfloat16)
    gate = torch.randn((7, Nf), generator=g, device=cuda).to(torch.bfloat16)
    seq = M // 7
    assert seq * 7 == M
    indices = torch.randint(0, 7, (seq,), generator=g, device=cuda)
    indices[3], indices[seq // 2], indices[seq - 1] = -1, 7, 1 << 40
    plain, _ = xops.scaled_mm(qa, qw, sa, sw, bias, torch.bfloat16, N.ACT_NONE, False)
    want = xops.gate_residual(residual.reshape(7, seq, Nf), plain.reshape(7, seq, Nf), gate, indices).reshape(M, Nf)
    assert want[3].isnan().all() and want[seq - 1].isnan().all() and not want[4].isnan().any()
    for x, w, r, t in ((qa, qw, residual, gate),
                       (embed(qa, K + 48, 16), embed(qw, K + 64, 32), embed(residual, Nf + 24, 8), embed(gate, Nf + 40, 16)),
                       (qa, qw, embed(residual, Nf + 24, 1), embed(gate, Nf + 12, 0))):
        out = xops.scaled_mm_gate_residual(x, w, sa, sw, bias, r, t, indices)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))
