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


# one-tile blocks (two to a CU) and two-tile blocks (one to a CU), each with a last round that is full enough and one that is not
@pytest.mark.parametrize("M,K,N,whole", [
    (1, 4096, 32000, 1), (16, 2048, 32000, 1), (4, 8192, 32000, 1), (1, 6144, 49152, 1), (17, 2048, 32000, 0), (16, 2048, 16352, 0),
    (1, 512, 32000, 0), (1, 1216, 32000, 0), (1, 1280, 32000, 1), (1, 5120, 20480, 0), (16, 1792, 20480, 0), (1, 5120, 24576, 1),
    (11, 4096, 32000, 1), (5, 4096, 24576, 0), (16, 4096, 50304, 0), (16, 4096, 49152, 1), (11, 5120, 40960, 1), (11, 5120, 32000, 0),
    (11, 3072, 32000, 0), (11, 3072, 16384, 1), (11, 8192, 128256, 1), (1, 4100, 32000, 0),
])
def test_dense_head(M, K, N, whole):
    from tgis_amd import native

    assert native.load_library().tgis_dense_gemm_whole_operand(M, K, N, 0) == whole


# up to 256 rows: matrices whose 64-row passes are done first, and those where the tall kernel is; above, it always serves
@pytest.mark.parametrize("M,K,N,act,whole", [
    (128, 4096, 12288, 0, 0), (129, 4096, 12288, 0, 1), (256, 4096, 12288, 0, 1), (129, 2048, 2560, 0, 0), (256, 2048, 2560, 0, 0),
    (257, 2048, 2560, 0, 1), (192, 1024, 1024, 0, 0), (192, 3072, 5120, 0, 0), (256, 3072, 5120, 0, 1), (192, 2048, 6144, 0, 1),
    (256, 4096, 4096, 0, 0), (129, 11008, 4096, 0, 1), (129, 256, 128, 0, 1), (64, 4096, 22016, 2, 0), (65, 4096, 22016, 2, 1),
    (128, 2048, 11264, 2, 0), (129, 2048, 11264, 2, 1), (96, 1024, 5632, 2, 0), (300, 1024, 5632, 2, 1), (300, 4096, 4096, 1, 0),
])
def test_int4_tall(M, K, N, act, whole):
    from tgis_amd import native

    lib = native.load_library()
    assert lib.tgis_gptq_gemm_whole_sums(M, K, N, K // 128, 0, act) == whole
    assert lib.tgis_gptq_gemm_whole_sums(M, K, N, K // 128, 1, act) == 0  # act-order
    assert lib.tgis_gptq_gemm_whole_sums(M, K, N, K // 32, 0, act) == 0   # groups shorter than a k64-step


# past 3072 rows: row counts at which 256 x 256 tiles fill their rounds of 256 and are dealt evenly, or most of a single one over a long k, and others
@pytest.mark.parametrize("M,K,N,act,pays", [
    (257, 4096, 12288, 0, 1), (3072, 11008, 4096, 0, 1), (4096, 11008, 4096, 0, 0), (4097, 11008, 4096, 0, 1), (8192, 4096, 12288, 0, 0), (6000, 4096, 12288, 0, 1),
    (3841, 4096, 4096, 0, 0), (3840, 4096, 4096, 0, 0), (3584, 4096, 4096, 0, 1), (7168, 11008, 4096, 0, 1), (8192, 13824, 5120, 0, 1), (5120, 5632, 2048, 0, 0),
    (4864, 5632, 2048, 0, 1), (4865, 5632, 2048, 0, 0), (5120, 5056, 2048, 0, 1), (8192, 4096, 22016, 2, 1), (8193, 4096, 22016, 2, 0), (8193, 4096, 4000, 0, 0),
    (4800, 8192, 10240, 0, 1), (4376, 8192, 10240, 0, 0), (5700, 8192, 8192, 0, 1), (6500, 7168, 7168, 0, 1), (6700, 7168, 7168, 0, 0), (7203, 5120, 15360, 0, 1), (6000, 13824, 5120, 0, 1),
    (6264, 13824, 5120, 0, 0), (7459, 14336, 4096, 0, 1), (7459, 11008, 4096, 0, 0), (6000, 5120, 5120, 0, 0),
])
def test_int4_library(M, K, N, act, pays):
    from tgis_amd import native

    lib = native.load_library()
    assert lib.tgis_gptq_gemm_fused_pays(M, K, N, K // 64, 0, act) == pays
    assert lib.tgis_gptq_gemm_fused_pays(M, K, N, K // 64, 1, act) == 0          # act-order: up to 256 rows alone
    assert lib.tgis_gptq_gemm_fused_pays(256, K, N, K // 64, 1, act) == 1


# the dense prefill kernel: from 65 rows on where the streaming kernel's passes are more than one short round, past 256 where the library's tiles would
# leave the chip idle or an activation launch is saved
@pytest.mark.parametrize("M,K,N,act,pays", [
    (64, 2048, 2048, 0, 0), (65, 2048, 2048, 0, 0), (65, 4096, 4096, 0, 1), (256, 6144, 24576, 4, 1), (257, 6144, 24576, 4, 0), (1400, 2048, 2048, 0, 1), (1401, 2048, 2048, 0, 0),
    (500, 2048, 6144, 0, 1), (501, 2048, 6144, 0, 0), (100, 2040, 2048, 0, 0), (100, 2048, 1024, 0, 0), (100, 8192, 1024, 0, 1), (100, 8192, 1023, 0, 0), (300, 448, 2048, 0, 0), (200, 64, 2048, 0, 1), (512, 4096, 22016, 2, 0), (513, 4096, 22016, 2, 1), (300, 2048, 11264, 2, 1),
    (65, 320, 1280, 0, 1), (65, 320, 1280, 5, 0), (896, 3072, 5120, 0, 0), (700, 3072, 5120, 0, 1), (900, 24576, 6144, 0, 1), (1708, 24576, 6144, 0, 1), (1709, 24576, 6144, 0, 0), (2048, 18944, 3584, 0, 1), (1793, 20480, 5120, 0, 0), (1408, 28672, 7168, 0, 0), (1032, 28672, 7168, 4, 1), (1033, 28672, 7168, 4, 0), (1024, 24576, 7200, 0, 0), (1448, 24576, 6144, 5, 1), (1449, 24576, 6144, 5, 0), (1600, 24576, 6144, 0, 0), (1601, 24576, 6144, 0, 1), (1650, 24576, 5888, 0, 0), (1738, 28672, 5120, 0, 1), (1739, 28672, 5120, 0, 0), (2048, 24576, 4096, 0, 1), (2049, 24576, 4096, 0, 0), (1401, 24640, 4096, 0, 0), (1400, 24640, 4096, 0, 1), (2048, 32768, 2048, 0, 1), (1401, 32768, 2080, 0, 0), (1401, 16384, 2048, 0, 0), (1401, 11008, 4096, 0, 0), (600, 28672, 8192, 0, 0), (600, 4096, 28672, 2, 0),
    (8192, 2048, 11264, 2, 1), (8193, 2048, 11264, 2, 0), (100, 2048, 2048, 1, 0), (0, 2048, 2048, 0, 0),
])
def test_dense_tall(M, K, N, act, pays):
    from tgis_amd import native

    assert (native.load_library().tgis_dense_tall_bytes(M, K, N, act) >= 0) == bool(pays)


def test_dense_tall_operands():
    """What the library's linear takes and the kernel does not read is not its to serve: one dimension, three, columns or rows out of step."""
    import types

    import torch

    from tgis_amd import native

    w = types.SimpleNamespace(K=512, N=2048, plans={})
    serves = lambda x: native.dense_tall_bytes(x, w) >= 0
    x = torch.zeros(300, 512, dtype=torch.float16)
    assert serves(x)
    assert not any(map(serves, (x.flatten()[:512], x.view(300, 1, 512), x.view(100, 3, 512).transpose(1, 2), x.t().contiguous().t(), x.view(-1)[4:4 + 299 * 512].view(299, 512))))


def test_dense_tall_scratch():
    """Its scratch fits the workspace that projections share, which captured graphs hold the address of."""
    from tgis_amd import native

    lib = native.load_library()
    assert max(lib.tgis_dense_tall_bytes(M, K, N, 2) for M in range(65, 1500, 61) for K in (64, 1024, 5632, 24576) for N in (1024, 2048, 6400, 22016)) <= 48 << 20


# split sums of the dense prefill kernel: a second block on some CUs costs more than three quarters of a round, so the parts end within a whole one
@pytest.mark.parametrize("M,K,N,parts", [(128, 6144, 6144, 4), (100, 6144, 6144, 5), (160, 8192, 10240, 3), (256, 11008, 4096, 4), (65, 24576, 6144, 5), (128, 4096, 4096, 4)])
def test_dense_tall_parts(M, K, N, parts):
    from tgis_amd import native

    rows = -(-M // 32) * 32
    assert native.load_library().tgis_dense_tall_partial_bytes(M, K, N) == rows * N * 4 * parts


# ... and stay parts of the streaming kernel where its passes are one round of short blocks, more than half full
@pytest.mark.parametrize("M,K,N,serves", [(64, 4096, 4096, 0), (65, 2048, 2048, 0), (256, 2048, 2560, 1), (192, 2048, 2560, 0), (128, 1024, 1024, 1), (256, 1024, 1024, 0), (128, 4096, 1024, 1),
                                          (128, 2560, 1024, 0), (257, 4096, 4096, 0), (100, 4096, 1000, 0)])
def test_dense_tall_parts_or_passes(M, K, N, serves):
    from tgis_amd import native

    assert (native.load_library().tgis_dense_tall_partial_bytes(M, K, N) >= 0) == bool(serves)


# phases of the x of several products in one launch: halved where that lets a CU take a second of more tiles than there are CUs
@pytest.mark.parametrize("M,K,N,k", [
    (21, 2048, 256 * 32, 1024), (21, 2048, 256 * 32 + 1, 512), (32, 4096, 130 * 32, 1024), (32, 4096, 516 * 32, 512), (17, 2048, 258 * 32, 1024), (21, 1024, 516 * 32, 1024),
    (16, 8192, 97 * 32, 2048), (16, 4096, 516 * 32, 1024), (8, 4096, 516 * 32, 2048), (16, 2048, 516 * 32, 2048), (33, 4096, 516 * 32, 512), (64, 512, 32, 512),
])
def test_dense_groups_phase(M, K, N, k):
    from tgis_amd import native

    assert native.load_library().tgis_dense_gemm_groups_phase(M, K, N) == k


# int4 launches in fragment order: blocks of 16 rows, but four for three where a wave walks one or two k64-steps of two tiles
@pytest.mark.parametrize("M,K,N,act,rows", [
    (1, 2048, 2048, 0, 16), (16, 2048, 2048, 0, 16), (17, 2048, 2048, 0, 32), (33, 2048, 2048, 0, 64), (48, 1024, 3072, 0, 64), (48, 4096, 4096, 0, 64), (33, 6144, 4096, 0, 48),
    (33, 4160, 4096, 0, 48), (48, 5632, 2048, 0, 64), (48, 4096, 12288, 0, 48), (48, 4096, 22016, 2, 48), (48, 1024, 8192, 2, 64), (48, 1024, 4096, 2, 48), (49, 4096, 12288, 0, 64), (64, 2048, 2048, 0, 64),
])
def test_int4_fragment_rows(M, K, N, act, rows):
    from tgis_amd import native

    assert native.load_library().tgis_gptq_fragment_rows(M, K, N, act) == rows
