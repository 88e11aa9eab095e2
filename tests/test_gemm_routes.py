"""CPU: which form of a GEMM the library chooses on each side of its rules (host-side queries, no compute)."""
import pytest


# the chip holds a block of every two tiles at once from 256 to 512 tiles; K: what fits in flight, and is worth it
@pytest.mark.parametrize("M,K,N,whole", [
    (32, 2048, 11264, 0), (33, 2048, 11264, 1), (64, 2048, 11264, 1), (65, 2048, 11264, 0),
    (48, 2048, 8160, 0), (48, 2048, 8192, 1), (48, 2048, 16384, 1), (48, 2048, 16416, 0), (48, 2048, 24576, 0), (48, 2048, 512, 0),
    (48, 1088, 11264, 0), (48, 1152, 11264, 1), (48, 2112, 11264, 0), (48, 256, 24576, 0), (48, 2000, 11264, 0),
])
def test_dense_gate_up(M, K, N, whole):
    from tgis_amd import native

    assert native.load_library().tgis_dense_gemm_whole_operand(M, K, N, 2) == whole
