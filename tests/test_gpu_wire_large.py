"""The FP8 wire decoder past the last-level cache, where its output stores are non-temporal."""
import pytest
import torch

import xgen_amd  # noqa: F401
from xgen_amd import _native as N
from xgen_amd.phaa import fp8_transport as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode_past_the_last_level_cache(cuda, dtype):
    """A decode that moves more than 256 MB (non-temporal output stores) gives the bytes of its peers'
    blocks decoded one by one (ordinary stores), and its strided form the same values in the gather's
    [head, position] order; widths whose outputs take 16-byte stores."""
    peers, seq, heads, dim, streams = 8, 14500, 2, 128, 3
    rows = seq * heads
    assert streams * peers * rows * (dim * 3 + 4) > 256 << 20
    g = torch.Generator(device=cuda).manual_seed(17)
    views = tuple(torch.randn((peers, seq, 1, heads, dim), generator=g, device=cuda).to(dtype) for _ in range(streams))
    wire, pad = T.encode_wire(views, dim, peers)
    outs = tuple(torch.empty((peers * rows, dim), dtype=dtype, device=cuda) for _ in range(streams))
    T.decode_wire(wire, outs, dim, peers, pad)
    block = wire.reshape(peers, -1)
    one = tuple(torch.empty((rows, dim), dtype=dtype, device=cuda) for _ in range(streams))
    for p in range(peers):
        T.decode_wire(block[p].clone(), one, dim, 1, pad)
        for o, w in zip(outs, one):
            assert torch.equal(o[p * rows:(p + 1) * rows].view(torch.int16), w.view(torch.int16))
    gathered = tuple(torch.full((heads, peers * seq, dim), 7.0, dtype=dtype, device=cuda) for _ in range(streams))
    strides = (N._c_i64 * 4)(seq * dim, dim, 0, peers * seq * dim)
    N.check(N.lib().xgen_fp8_wire_decode_strided(
        N.dtype_code(dtype), streams, wire.data_ptr(), peers, seq, 1, heads, dim, strides, peers * seq - 3,
        *(t.data_ptr() for t in gathered), N.stream_of(wire)), "xgen_fp8_wire_decode_strided")
    for t, o in zip(gathered, outs):
        want = o.reshape(peers, seq, heads, dim).permute(2, 0, 1, 3).reshape(heads, peers * seq, dim).clone()
        want[:, -3:] = 7.0  # positions past the valid length are not written
        assert torch.equal(t.view(torch.int16), want.view(torch.int16))
