"""Weight gradients at the edges of their kernel's 4 x 64 pixel tiles and for every pair of channel
counts, against the oracle (bf16 storage emulated).  Tolerance: the per-layer bound of the U-Net tests,
1e-2 relative L2 (bf16 roundings at boundaries; a wrong tap, channel, pixel or tile is O(1))."""
import numpy as np
import pytest

from oracle import unet as OU

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,ch,c_in,c_out,relu", [
    (4, 64, (16, 64), 1, 1, 1), (5, 65, (16, 64), 2, 2, 1), (3, 63, (16, 32), 1, 2, 0), (9, 129, (16, 16), 2, 1, 1),
    (8, 127, (16, 32, 64), 1, 1, 0), (13, 7, (16, 64, 32), 1, 1, 1), (130, 3, (16, 64), 2, 1, 1)])
def test_weight_gradients_at_tile_edges(torch_gpu, H, W, ch, c_in, c_out, relu):
    torch = torch_gpu
    from autopdex_amd.learned import UNetPreconditioner
    from tests.test_gpu_unet import _bf16_bits, _copy
    B, L = 3, len(ch)
    print(f"[case] wgrad {H}x{W} {ch} {c_in} {c_out} relu={relu}", flush=True)
    net = UNetPreconditioner(H, W, L, ch, c_in, c_out, relu=bool(relu), batch=B, seed=2)
    rng = np.random.default_rng(H * 1000 + W)
    theta = net.get_params()
    x = rng.standard_normal((B, H, W, c_in)).astype(np.float32)
    xb = torch.from_numpy(_bf16_bits(x).view(np.int16)).cuda()
    _copy(net.buffers()[0], xb.data_ptr(), xb.numel() * 2)
    net.forward()
    t = rng.standard_normal((B, H, W, c_out)).astype(np.float32)
    net.loss_backward(torch.from_numpy(t.ravel()).cuda())
    g = net.get_grads()
    orc = OU.UNetOracle(L, ch, c_in, c_out, relu, H, W, bf16_storage=True)
    orc.forward(theta.astype(np.float64), OU.bf16(x))
    _, ref = orc.loss_backward(t.astype(np.float64))
    for name, (w_off, b_off, ci, co, cop, wk) in orc.layout.items():
        gw, gr = g[w_off:b_off + co], ref[w_off:b_off + co]
        assert np.linalg.norm(gw - gr) <= 1e-2 * np.linalg.norm(gr), name
