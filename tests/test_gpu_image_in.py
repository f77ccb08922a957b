"""mr_image_in_f32 (both copies of a segment's image input in one pass) and the gapless row
quantizer, bit for bit against the oracle's cast, transpose and quantize_activation."""
import numpy as np
import pytest
import torch

from mira_amd import _lib as L
from mira_amd import pack
from oracle import golden as G

from conftest import bits_equal
from gpu_util import T, empty, stream, sync

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("n,c,h,w,i8", [(1, 1, 1, 1, True), (2, 3, 5, 7, True), (1, 64, 8, 8, True), (3, 65, 9, 15, True),
                                        (1, 130, 3, 43, False), (37, 128, 28, 28, True), (2, 63, 64, 65, True)])
def test_image_in(lib, n, c, h, w, i8, f16):
    rng = np.random.default_rng(n + c + h)
    x = (rng.standard_normal((n, c, h, w)) * 3).astype(np.float32)
    x.flat[0] = np.inf
    x.flat[-1] = -70000.0                 # overflows f16
    cp, xs = pack.c_pad_for(c), 0.0371
    d = T(x)
    y, q = empty((n, h, w, c), torch.float32), empty((n, h, w, cp), torch.int8)
    q.fill_(77)
    L.check(lib.mr_image_in_f32(d.data_ptr(), n, c, h, w, int(f16), y.data_ptr(), q.data_ptr() if i8 else None, cp, xs,
                                stream()), "image_in")
    sync()
    with np.errstate(over="ignore"):
        want = (x.astype(np.float16).astype(np.float32) if f16 else x).transpose(0, 2, 3, 1)
    assert bits_equal(y.cpu().numpy(), np.ascontiguousarray(want))
    if i8:
        wq = np.zeros((n, h, w, cp), np.int8)
        wq[..., :c] = G.quantize_activation(want, np.float32(xs)).astype(np.int8)
        assert bits_equal(q.cpu().numpy(), wq)
    assert bits_equal(d.cpu().numpy(), x)          # the input is left as it was


@pytest.mark.parametrize("rows,cols,ldx", [(1, 16, 16), (3, 16, 16), (5, 1040, 1040), (64, 48, 52), (7, 20, 20)])
def test_quantize_rows_gapless(lib, rows, cols, ldx):
    """ldx == cols == ldq takes the flat kernel; the last two (a row gap, padded rows) do not."""
    rng = np.random.default_rng(rows)
    x = (rng.standard_normal((rows, ldx)) * 4).astype(np.float32)
    x[0, :3] = np.inf, -np.inf, 2.5 * np.float32(0.031)
    ld = pack.row_stride_for(cols)
    d, q = T(x), empty((rows, ld), torch.int8)
    L.check(lib.mr_quantize_rows(d.data_ptr(), rows, cols, ldx, q.data_ptr(), ld, 0.031, stream()), "quantize")
    sync()
    want = np.zeros((rows, ld), np.int8)
    want[:, :cols] = G.quantize_activation(x[:, :cols], np.float32(0.031)).astype(np.int8)
    assert bits_equal(q.cpu().numpy(), want)
