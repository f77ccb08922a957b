"""Small results: the K-split int8 tiles (qrows) and the small expansion + depthwise tiles, against
the oracle, at the edges of their tiles and on both sides of the rules that choose them."""
import pytest

import test_gpu_kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,h,w,o,k,s,p,d", [
    (1, 64, 3, 3, 1, 3, 1, 1, 1),         # 9 rows, one column
    (1, 512, 7, 7, 512, 3, 1, 1, 1),      # 16 x 16 tiles, 72 steps
    (1, 65, 9, 5, 33, 3, 2, 1, 1),        # channels padded to 80: chunks of 16 bytes span taps within a step
    (2, 16, 14, 14, 17, 5, 1, 4, 2),      # 16 channels (one chunk per tap), dilation, wide padding
    (1, 130, 11, 13, 40, 1, 2, 0, 1),     # 1x1, stride 2
    (1, 704, 5, 5, 48, 3, 1, 0, 1),       # 99 steps: past three batches of a wave's loads
    (1, 64, 56, 56, 64, 3, 1, 1, 1),      # 16 x 32 tiles
    (2, 64, 64, 64, 32, 3, 1, 1, 1),      # 32 x 32 tiles, the largest grid for 9 steps
    (2, 64, 64, 65, 32, 3, 1, 1, 1),      # one tile more: qgemm's tiles
])
def test_small_convolutions(lib, n, c, h, w, o, k, s, p, d):
    K.test_qconv2d(lib, n, c, h, w, o, k, s, p, d)


@pytest.mark.parametrize("M,K_,N", [(9, 65, 1), (16, 2048, 16), (17, 2112, 33), (33, 128, 1000), (64, 576, 4096),
                                    (65, 512, 512), (1024, 640, 250), (64, 4096, 4128)])
def test_small_matmuls(lib, M, K_, N):
    K.test_qmatmul_bias_relu_requant(lib, M, K_, N)


@pytest.mark.parametrize("n,k,c,h,s,f32_out", [
    (1, 24, 144, 29, 2, True), (1, 96, 576, 14, 2, False), (1, 160, 960, 15, 2, False),    # 4 x 4 tiles, stride 2
    (1, 32, 192, 28, 1, True), (2, 96, 576, 15, 1, False),                                # 7 x 7 tiles, stride 1
    (30, 24, 96, 28, 1, False), (30, 24, 96, 28, 2, False),                                # enough for 14 / 7
])
def test_expand_dw_tiles(lib, n, k, c, h, s, f32_out):
    K.test_qconv1x1_dw3x3(lib, n, k, c, h, s, f32_out)


@pytest.mark.parametrize("n,cin,c,h,ss,s", [(1, 3, 32, 64, 2, 1), (30, 3, 96, 60, 2, 1), (30, 3, 32, 60, 1, 2)])
def test_stem_tiles(lib, n, cin, c, h, ss, s):
    K.test_qstem3x3_dw3x3(lib, n, cin, c, h, ss, s)
