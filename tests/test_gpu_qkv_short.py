"""QKV projection of short prompts (launch_qkv_gemm, kernels.hpp:29-36, up to 256
tokens): every tile of csrc/qkv_short.hip at its edges, against the product in
64 bits and, fused, against the two launches bit for bit."""
import numpy as np
import pytest

from test_gpu_qkv_gemm import fused_case, rand_inputs, run_gemm

pytestmark = pytest.mark.gpu


# one token tile and several of each tile size, token and feature remainders (N
# odd, N below one head, N not a multiple of 128), K of one unit more than the
# waves share evenly
@pytest.mark.parametrize("M,N,K", [
    (1, 3072, 2048), (16, 3072, 1024), (17, 3072, 2048), (32, 3072, 1088), (33, 3072, 2048),
    (64, 3072, 2048), (65, 3072, 1088), (128, 3072, 2048), (129, 3072, 1024), (255, 3072, 2048),
    (256, 3072, 1088), (256, 6144, 1024), (5, 131, 1024), (40, 24, 1152), (200, 1000, 2112),
    (256, 1536, 4096), (70, 200, 1984)])
def test_short_prompt_tiles(attn, gpu, M, N, K):
    print(f"[case] short M={M} N={N} K={K}", flush=True)
    x, w = rand_inputs(M, N, K, 7 * M + N + K)
    y = run_gemm(attn, gpu, x, w).view(np.float16).astype(np.float64)
    xf, wf = (t.view(np.float16).astype(np.float64) for t in (x, w))
    exact = xf @ wf.T
    # fp16 rounding of the result plus the fp32 sums' bound, K steps of 2^-24 of
    # the terms' magnitudes (the products of fp16 values are exact in fp32)
    bound = 2.0 ** -11 * np.abs(exact) + K * 2.0 ** -24 * (np.abs(xf) @ np.abs(wf).T) + 2.0 ** -24
    assert (np.abs(y - exact) <= bound).all()


@pytest.mark.parametrize("M,start_pos,rotate", [(1, 0, True), (16, 31, True), (17, 2, False),
                                                (31, 0, True), (64, 9, True), (97, 1, True),
                                                (193, 0, True), (256, 300, False)])
@pytest.mark.parametrize("Hq,Hkv", [(16, 4), (3, 1)])
def test_short_prompt_fused_bitexact(attn, gpu, M, start_pos, rotate, Hq, Hkv):
    print(f"[case] short fused M={M} pos={start_pos} rotate={rotate} {Hq}/{Hkv}", flush=True)
    fy, fc, ty, tc, _ = fused_case(attn, gpu, M, start_pos, rotate, Hq, Hkv)
    assert np.array_equal(fy, ty), "y"
    assert np.array_equal(fc, tc), "cache"


# head_dim 64, an odd and an even number of heads, each tile
@pytest.mark.parametrize("M,start_pos,rotate", [(1, 5, True), (16, 0, True), (17, 3, False),
                                                (33, 0, True), (64, 7, True), (97, 1, True),
                                                (130, 0, True), (256, 9, True)])
@pytest.mark.parametrize("Hq,Hkv", [(16, 4), (3, 1), (32, 8), (5, 1)])
def test_short_prompt_fused_64_dim_heads_bitexact(attn, gpu, M, start_pos, rotate, Hq, Hkv):
    print(f"[case] short fused d64 M={M} pos={start_pos} {Hq}/{Hkv}", flush=True)
    fy, fc, ty, tc, _ = fused_case(attn, gpu, M, start_pos, rotate, Hq, Hkv, 64, 1024)
    assert np.array_equal(fy, ty), "y"
    assert np.array_equal(fc, tc), "cache"


# where the rounds of the short tiles cost more than those of the tiles for longer
# prompts (256 CUs), the latter run: their bits are those of any of them
@pytest.mark.parametrize("M,N,short", [(128, 6144, True), (192, 6144, False), (256, 6144, False),
                                       (64, 9216, True), (192, 9216, False), (256, 12288, False),
                                       (32, 18432, True), (64, 18432, False), (128, 18432, False)])
def test_short_tiles_only_where_cheaper(attn, gpu, M, N, short):
    print(f"[case] short or long M={M} N={N}", flush=True)
    x, w = rand_inputs(M, N, 1024, M + N)
    y = run_gemm(attn, gpu, x, w)
    try:
        attn.set_option("qkv_gemm_tokens_per_wave", 64)
        ref = run_gemm(attn, gpu, x, w)
    finally:
        attn.set_option("qkv_gemm_tokens_per_wave", 0)
    assert np.array_equal(y, ref) != short
