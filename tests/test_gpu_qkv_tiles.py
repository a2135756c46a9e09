"""The prefill projection's tiles above 256 tokens: whichever one the rounds of
workgroups pick, the bits are those of the 128 x 128 tile (every tile adds the
k-values in one order), and the fused epilogue equals the two launches."""
import numpy as np
import pytest
import torch

from test_gpu_qkv_gemm import check_vs_oracle, dev, fused_case, host, rand_inputs

pytestmark = pytest.mark.gpu


def run_gemm(attn, gpu, x, w):
    # Y at the start of an allocation: the wide tiles want 16-byte rows
    (M, K), N = x.shape, w.shape[0]
    y = torch.full((M, N), float("nan"), dtype=torch.float16, device=gpu)
    attn.qkv_gemm(dev(x, gpu), y, dev(w, gpu), M, K, N)
    torch.cuda.synchronize()
    return host(y)


# both sides of the picks at 256 CUs and N = 3072: 64 tokens a tile to 640, 128
# to 1280, 256 to 2560, 128 to 2688, 256 x 256 to 5376, 256 x 384 beyond; K of
# one to four stages
@pytest.mark.parametrize("M,N,K", [
    (257, 3072, 128), (640, 3072, 64), (641, 3072, 192), (1280, 3072, 128), (1281, 3072, 256),
    (2560, 3072, 64), (2561, 3072, 192), (2689, 3072, 128), (5376, 3072, 192), (5377, 3072, 64),
    (4097, 2048, 256), (9000, 1024, 64), (300, 1000, 2048), (3000, 1280, 2048)])
def test_automatic_tile_identical(attn, gpu, M, N, K):
    print(f"[case] tiles M={M} N={N} K={K}", flush=True)
    x, w = rand_inputs(M, N, K, M + N + K)
    auto = run_gemm(attn, gpu, x, w)
    try:
        attn.set_option("qkv_gemm_tokens_per_wave", 64)
        ref = run_gemm(attn, gpu, x, w)
    finally:
        attn.set_option("qkv_gemm_tokens_per_wave", 0)
    assert np.array_equal(auto, ref)
    check_vs_oracle(auto, x, w, np.unique(np.r_[0, M - 1, np.arange(0, M, 97)]))


@pytest.mark.parametrize("M,start_pos,rotate", [(640, 3, True), (1200, 0, False), (2600, 1, True),
                                                (3333, 17, True)])
def test_automatic_tile_fused_bitexact(attn, gpu, M, start_pos, rotate):
    print(f"[case] fused tiles M={M} pos={start_pos} rotate={rotate}", flush=True)
    fy, fc, ty, tc, _ = fused_case(attn, gpu, M, start_pos, rotate, K=192)
    assert np.array_equal(fy, ty) and np.array_equal(fc, tc)


# head_dim 64: two heads to a 128-feature tile, the last one alone where
# Hq + 2 Hkv is odd; each tile; both sides of the short prompts
@pytest.mark.parametrize("Hq,Hkv", [(16, 4), (3, 1), (5, 1), (8, 8)])
@pytest.mark.parametrize("M,start_pos,rotate", [(256, 0, True), (257, 9, True), (1300, 3, False),
                                                (3333, 2, True), (6000, 0, True)])
def test_fused_64_dim_heads_bitexact(attn, gpu, Hq, Hkv, M, start_pos, rotate):
    print(f"[case] fused d64 {Hq}/{Hkv} M={M} pos={start_pos} rotate={rotate}", flush=True)
    fy, fc, ty, tc, _ = fused_case(attn, gpu, M, start_pos, rotate, Hq, Hkv, 64, 192)
    assert np.array_equal(fy, ty) and np.array_equal(fc, tc)


def test_fused_64_dim_heads_wide_tile(attn, gpu):
    try:
        attn.set_option("qkv_gemm_wide", 2)
        fy, fc, ty, tc, _ = fused_case(attn, gpu, 700, 5, True, 16, 4, 64, 192)
    finally:
        attn.set_option("qkv_gemm_wide", 0)
    assert np.array_equal(fy, ty) and np.array_equal(fc, tc)
