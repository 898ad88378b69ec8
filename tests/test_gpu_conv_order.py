"""The forward convolution's tile order where dil planes are few row groups: one
(a block of one group), a number that 16 does not divide (equal blocks), and one
that does, with partial last groups and turns.  Against the convolution oracle, FP32
outputs to 1e-5 of their scale (sums of exact BF16 products in another order)."""
import numpy as np
import pytest

import conv_oracle as co
import qmin
from test_gpu_warmstart import check, dev_bf16, ptr, stream

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("lx,ly,lz,dil", [(16, 16, 40, 1), (16, 5, 30, 2), (16, 40, 17, 7), (90, 17, 5, 1), (64, 16, 9, 4),
                                          (16, 64, 11, 3)])
def test_every_tile_is_computed(lx, ly, lz, dil):
    rng = np.random.default_rng(lx + ly)
    n = lx * ly * lz
    x, w = co.bf16_round(rng.normal(size=(n, 16))), co.bf16_round(rng.normal(size=(27, 16, 16)) * 0.2)
    ref = co.forward(x, w, np.zeros(16), (lx, ly, lz), dil, relu_in=False)
    xd, wd = dev_bf16(x), dev_bf16(w)
    y = torch.full((n * 16,), float("nan"), dtype=torch.float32, device="cuda")
    check(qmin.library().qm_ws_conv_forward(ptr(xd), 16, ptr(wd), None, 16, None, None, ptr(y), lx, ly, lz, dil, 0,
                                            stream()))
    torch.cuda.synchronize()
    np.testing.assert_allclose(y.cpu().numpy().reshape(n, 16), ref, rtol=0, atol=1e-5 * np.abs(ref).max())
