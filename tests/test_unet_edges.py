"""U-net convolutions and gradients (GPU) where their work split can go wrong:
every count of 16-channel tiles, channels that end inside a tile and inside a
group of 8, volumes that end inside a brick (16 x 4 x 4 voxels), more bricks
than weight-gradient blocks.  Every weight and bias tensor's gradient is
compared on its own with the FP64 restatement.

The restatement rounds every stored tensor to bf16 as the kernels do; what is
left is the FP32 accumulation order and values that round to neighbouring bf16
numbers (2^-8 apart, a small fraction of them): relative L2 error <= 1e-2 per
tensor.  A lost or doubled tap, channel, voxel or partial is of order one."""
import numpy as np
import pytest

from oracle import unet_ref
from test_unet import _bf16, _rel2, _weights_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channels,cin,dims,N", [
    ((1,), 1, (1, 1, 1), 1), ((7,), 3, (3, 5, 17), 2), ((17,), 9, (5, 4, 16), 1),
    ((33,), 17, (4, 9, 31), 1), ((49,), 25, (6, 3, 15), 1), ((64,), 33, (4, 4, 16), 2),
    ((16, 64), 2, (4, 8, 34), 1), ((12,), 2, (16, 16, 48), 17)])
def test_every_gradient_tensor(channels, cin, dims, N):
    import torch
    from ifem_amd import Session
    print(f"[gpu] unet edges channels={channels} cin={cin} dims={dims} N={N}", flush=True)
    (D, H, W), L, cout = dims, len(channels), 2
    rng = np.random.default_rng(17)
    x = _bf16(rng.standard_normal((N, cin, D, H, W)).astype(np.float32))
    t = rng.standard_normal((N, cout, D, H, W)).astype(np.float32)
    with Session() as s:
        s.unet_create(L, channels, cin, cout, seed=7)
        p = s.unet_params()
        p = p + 0.05 * rng.standard_normal(p.shape).astype(np.float32)
        s.unet_set_params(p)
        xd, td = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
        yd = torch.empty((N, cout, D, H, W), dtype=torch.float32, device="cuda")
        s.unet_forward(xd.data_ptr(), yd.data_ptr(), N, D, H, W)
        torch.cuda.synchronize()
        _, g = s.unet_gradient(xd.data_ptr(), td.data_ptr(), N, D, H, W)
        y = yd.cpu().numpy()
    pq = _weights_bf16(p, L, channels, cin, cout).astype(np.float64)
    yr, _, gr = unet_ref.forward_backward(pq, x, t, L, list(channels), cin, cout,
                                          quant=lambda v: _bf16(v).astype(np.float64))
    assert _rel2(y, yr) <= 1e-2
    for ci, co, _, w, b in unet_ref.layout(L, list(channels), cin, cout)[0]:
        assert _rel2(g[w:w + co * ci * 27], gr[w:w + co * ci * 27]) <= 1e-2, (ci, co)
        assert _rel2(g[b:b + co], gr[b:b + co]) <= 1e-2, (ci, co)
