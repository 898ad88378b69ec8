"""Warm-start convolutions at the edges of their tiles: rows cut into segments
with a halo, rows shorter and longer than a work-group's 256 sites, dilations
that no halo holds or that exceed the row, partial last work-groups, and buffers
that are not 16-byte aligned.  Against the convolution oracle.

Tolerances as for the other convolution tests: FP32 sums of exact BF16 products
in another order than the oracle, 1e-5 of the output scale; BF16 outputs one
rounding more (2^-8 relative).
"""
import numpy as np
import pytest

import conv_oracle as co
import qmin
from test_gpu_warmstart import check, dev_bf16, host_bf16, ptr, stream

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# whole rows; segments with a halo; a row longer than 256; a dilation that fits no
# halo (each tap staged by itself); a dilation above the row; one-site rows
TILES = [(24, 11, 3, 1), (75, 5, 4, 1), (130, 3, 3, 8), (203, 2, 3, 4), (300, 2, 3, 8), (400, 3, 2, 160), (5, 7, 3, 11),
         (1, 9, 6, 2)]


def offset(t, k):
    """A copy of t that starts k elements into its allocation."""
    b = torch.empty(t.numel() + k, dtype=t.dtype, device="cuda")
    b[k:].copy_(t.reshape(-1))
    return b[k:]


@pytest.mark.parametrize("lx,ly,lz,dil", TILES)
@pytest.mark.parametrize("cin,cout", [(16, 32), (32, 64), (64, 16), (64, 64)])
@pytest.mark.parametrize("shift", [0, 4])
def test_forward_tiles(lx, ly, lz, dil, cin, cout, shift):
    lib = qmin.library()
    rng = np.random.default_rng(lx + dil + cin)
    dims, n = (lx, ly, lz), lx * ly * lz
    x = co.bf16_round(rng.normal(size=(n, cin)))
    w = co.bf16_round(rng.normal(size=(27, cout, cin)) * 0.2)
    b = rng.normal(size=cout).astype(np.float32).astype(np.float64)
    mask = co.bf16_round(rng.normal(size=(n, cout)))
    ref = co.forward(x, w, b, dims, dil, relu_in=True)
    xd, wd, md = dev_bf16(x), dev_bf16(w), dev_bf16(mask)
    yb = torch.empty(n * cout, dtype=torch.int16, device="cuda")
    if shift:   # weights 8-byte aligned, the input too where it takes 8-byte loads; outputs 2-byte aligned
        xd = offset(xd, 4) if cin < 64 else xd
        wd, md, yb = offset(wd, 4), offset(md, 1), offset(yb, 1)
    bd = torch.from_numpy(b.astype(np.float32)).cuda()
    yf = torch.empty(n * cout, dtype=torch.float32, device="cuda")
    check(lib.qm_ws_conv_forward(ptr(xd), cin, ptr(wd), ptr(bd), cout, None, None, ptr(yf), lx, ly, lz, dil, 1,
                                 stream()))
    check(lib.qm_ws_conv_forward(ptr(xd), cin, ptr(wd), ptr(bd), cout, ptr(md), ptr(yb), None, lx, ly, lz, dil, 1,
                                 stream()))
    torch.cuda.synchronize()
    tol = 1e-5 * np.abs(ref).max()
    np.testing.assert_allclose(yf.cpu().numpy().reshape(n, cout), ref, rtol=0, atol=tol)
    np.testing.assert_allclose(host_bf16(yb).reshape(n, cout), np.where(mask > 0, ref, 0.0), rtol=2 ** -8, atol=tol)


@pytest.mark.parametrize("lx,ly,lz,dil", TILES + [(16, 4, 5, 8), (64, 3, 2, 4)])
@pytest.mark.parametrize("cin,cout", [(16, 32), (32, 64), (64, 16), (64, 64)])
@pytest.mark.parametrize("chunk,shift", [(64, 0), (4096, 1)])
def test_weight_and_bias_gradient_pieces(lx, ly, lz, dil, cin, cout, chunk, shift):
    """Rows that are no multiple of eight sites, pieces that wrap around a row,
    several slots and one, and buffers of four-byte alignment."""
    lib = qmin.library()
    rng = np.random.default_rng(lx + dil + cout)
    dims, n = (lx, ly, lz), lx * ly * lz
    x, g = co.bf16_round(rng.normal(size=(n, cin))), co.bf16_round(rng.normal(size=(n, cout)))
    ref = co.weight_grad(g, x, dims, dil, relu_in=True)
    chunks = (n + chunk - 1) // chunk
    part = offset(torch.empty(chunks * 27 * cout * cin, dtype=torch.float32, device="cuda"), shift)
    dw = torch.empty(27 * cout * cin, dtype=torch.float32, device="cuda")
    gd, xd = dev_bf16(g), dev_bf16(x)
    check(lib.qm_ws_conv_wgrad(ptr(gd), cout, ptr(xd), cin, 1, lx, ly, lz, dil, ptr(part), chunk, ptr(dw), stream()))
    db = torch.empty(cout, dtype=torch.float32, device="cuda")
    bpart = torch.empty(37 * cout, dtype=torch.float32, device="cuda")
    gb = offset(gd, shift)
    check(lib.qm_ws_bias_grad(ptr(gb), n, cout, ptr(bpart), 37, ptr(db), stream()))
    torch.cuda.synchronize()
    np.testing.assert_allclose(dw.cpu().numpy().reshape(27, cout, cin), ref, rtol=0, atol=1e-5 * np.abs(ref).max())
    np.testing.assert_allclose(db.cpu().numpy(), g.sum(axis=0), rtol=1e-5, atol=1e-5 * np.sqrt(n))
