"""The output tile that a W8A8 GEMM call runs on (xgen_amd/csrc/gemm_tile.hip: choose_gemm_tile), asked of
the built library on the host.  Without a device it counts 256 CUs, an MI355X's."""
import pytest

from conftest import GEMM_KINDS, gemm_tile

LARGE = (256, 256)


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("kind", sorted(GEMM_KINDS))
@pytest.mark.parametrize("K", [16, 64, 128, 256])
@pytest.mark.parametrize("M,Nf", [(8192, 9216), (15624, 3072), (15624, 18432), (31248, 9216), (66048, 16384)])
def test_many_rows_of_short_k_stay_on_the_large_kernel(built_library, M, Nf, K, kind, gated):
    """A smaller tile takes as many K steps as it has slots, whatever K: 32 x 128 measured up to 3.8
    times the 256 x 256 kernel's time on these."""
    assert gemm_tile(kind, M, Nf, K, gated) == LARGE


@pytest.mark.parametrize("kind,M,Nf,K,gated,tile", [
    ("fp8_exact", 256, 1024, 1024, False, (32, 64)),     # latency: as many workgroups as there are CUs
    ("int8", 2, 18432, 3072, False, (32, 128)),
    ("fp8_exact", 1003, 3072, 3072, False, (128, 128)),
    ("fp8", 1955, 12288, 3072, False, (256, 192)),
    ("fp8", 1955, 3072, 12288, False, (128, 192)),
    ("fp8", 3906, 3072, 3072, True, (256, 192)),
    ("fp8", 15624, 9216, 3072, False, LARGE),
    ("int8", 15624, 12288, 3072, False, LARGE),
    ("fp8", 15624, 3072, 3072, True, LARGE),
    ("fp8_exact", 1955, 18432, 64, False, LARGE),        # short K: 10% below the large kernel or not at all
    ("fp8_exact", 100, 1024, 64, False, (32, 128)),      # few rows of short K leave it idle
    # shapes whose GPU tests are written for the large kernel: short tiles, row chunks
    ("fp8", 8192, 10240, 64, False, LARGE), ("fp8", 8192, 10240, 128, False, LARGE), ("fp8", 8192, 10240, 192, False, LARGE),
    *((kind, rows, 16384, 64, False, LARGE) for kind in ("fp8", "fp8_exact", "int8") for rows in (66048, 33024)),
    ("fp8", 66048, 16384, 64, True, LARGE), ("fp8", 33024, 16384, 64, True, LARGE),
])
def test_choice(built_library, kind, M, Nf, K, gated, tile):
    assert gemm_tile(kind, M, Nf, K, gated) == tile


@pytest.mark.parametrize("kind,M,Nf,K,plain,accumulators", [
    ("fp8_exact", 15624, 5376, 384, (256, 192), LARGE),  # the accumulators' stores: 228 us on 256 x 192, 148 there
    ("fp8", 13032, 5376, 7168, (256, 128), LARGE),
    ("fp8", 1955, 12288, 3072, (256, 192), (256, 192)),
    ("fp8_exact", 1003, 3072, 3072, (128, 128), (128, 128)),
])
def test_choice_with_accumulators(built_library, kind, M, Nf, K, plain, accumulators):
    assert gemm_tile(kind, M, Nf, K) == plain
    assert gemm_tile(kind, M, Nf, K, accumulators=True) == accumulators
