"""What the library's own choice runs for a shape (the plan queries need no GPU): the lines that the
sources draw from measured times, on both sides."""

import pytest

from kernels import fp8, fused, w4a16


@pytest.mark.parametrize("M,N,K", [(1030, 1012, 2048), (130, 17924, 1024), (200, 4096, 14336), (161, 6144, 4096),
                                   (256, 8064, 2560)])
def test_int4_rows_stay_on_the_row_blocks(M, N, K):
    """N % 8 == 4, and up to 256 rows on narrow weights: the blocks round no weight, the GEMM rounds
    each to fp16."""
    assert w4a16.config_for(M, N, K).startswith("mfma,")
    assert w4a16.kernel_name(M, N, K).startswith("w4a16_mfma_kernel<")


@pytest.mark.parametrize("M,N,K", [(1, 14336, 4096), (1, 8064, 11008), (1, 151936, 1536), (2, 40960, 2560), (2, 28672, 4096)])
def test_int4_one_and_two_rows_stay_on_the_valu_kernel(M, N, K):
    """However large the weights: its error is the smaller, and the quantized lm_head and most other
    shapes are slower on the MFMA kernel."""
    assert w4a16.config_for(M, N, K).startswith("valu,")


@pytest.mark.parametrize("N,K,fuses", [(8192, 8192, True), (24576, 1024, True), (65536, 512, True), (20480, 1536, True),
                                       (24576, 2048, True), (28672, 1536, False), (12288, 4096, False),
                                       (17920, 2560, False), (151936, 1024, False), (151936, 1536, False)])
def test_one_row_norm_in_the_projections_launch(N, K, fuses):
    assert fused.norm_fuses(N, K) == fuses


@pytest.mark.parametrize("M,N,K,path", [(33, 2048, 13312, "mfma"), (48, 3072, 8192, "mfma"), (64, 2560, 13312, "mfma"),
                                        (65, 1536, 14336, "mfma"), (128, 1536, 13312, "mfma"), (140, 1536, 13312, "gemm"),
                                        (33, 4096, 14336, "gemm"), (96, 2048, 12288, "gemm"), (33, 6144, 4096, "gemm"),
                                        (48, 1028, 20480, "mfma"), (65, 1028, 20480, "gemm"), (64, 1544, 14336, "mfma"),
                                        (65, 1544, 14336, "gemm"), (48, 2052, 10240, "gemm")])
def test_e4m3_hand_over_to_the_gemm_on_large_narrow_weights(M, N, K, path):
    """At 96 tiles of 128 columns x 16 rows; rows of less alignment at 60 and 36."""
    assert fp8.config_for(M, N, K).startswith(path + ",")


@pytest.mark.parametrize("M,N,K,plan", [(4, 7936, 2560, "block_n=64"), (13, 4096, 5632, "block_n=64"),
                                        (5, 5376, 4096, "block_n=64"), (2, 1536, 14336, "block_n=64"),
                                        (2, 5120, 4096, "block_n=128,split_k=6"), (4, 5120, 4096, "block_n=64"),
                                        (13, 4096, 7680, "block_n=128,split_k=8"), (13, 6144, 3584, "block_n=128,split_k=5"),
                                        (5, 17920, 7168, "block_n=128,split_k=5"), (12, 18688, 4096, "block_n=128,split_k=3"),
                                        (13, 17920, 4096, "block_n=128,split_k=1"), (5, 17920, 3072, "block_n=128,split_k=1"),
                                        (8, 22528, 7168, "block_n=128,split_k=1"), (13, 28672, 4096, "block_n=128,split_k=1"),
                                        (13, 4096, 14336, "block_n=128,split_k=8")])
def test_e4m3_decode_rows_on_large_weights(M, N, K, plan):
    """128-column tiles on at most one workgroup per CU, where the 64-column or split tiles do not
    fill the CUs in one round themselves."""
    assert fp8.config_for(M, N, K).startswith("mfma," + plan)
