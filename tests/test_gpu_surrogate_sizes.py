"""GPU: training kernels of the surrogate at batch sizes around their tiles.

A batch is cut into 64-point tiles (padding points must not count), tiles
are dealt to at most 256 workgroups (16,384 points: one each) and the weight
gradients to at most 64 point ranges of four tiles.
"""
import numpy as np
import pytest

from oracle import mlp_ref as M

pytestmark = pytest.mark.gpu

CS = np.array([0.3, -0.2, 0.1, 6.0])


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 1023, 16384, 16449])
def test_batch_sizes_match_oracle(n):
    import torch
    from gimic_amd.surrogate import Network
    g = torch.Generator(device="cuda").manual_seed(n)
    r = 12.0 * torch.rand((n, 3), generator=g, dtype=torch.float64, device="cuda") - 6.0
    t = torch.randn((n, 9), generator=g, dtype=torch.float64, device="cuda")
    scale = np.linspace(0.5, 2.0, 9)
    net = Network(1.5, CS, scale, seed=5)
    p, fr, rn, tn = net.params().astype(np.float64), net.freqs(), r.cpu().numpy(), t.cpu().numpy()
    print("case mlp batch of", n, flush=True)
    loss, grad = net.loss_grad(r, t, 0.05)
    l_emu, g_emu = M.loss_grad(p, fr, CS, scale, rn, tn, 0.05, bf=True)
    assert abs(loss - l_emu) <= 1e-4 * abs(l_emu)
    # a BF16 operand that rounds the other way moves a gradient by up to 2^-8
    # of one of its terms: the bound of a single weight block
    assert np.linalg.norm(grad - g_emu) <= M.GPU_BLOCK_TOL * np.linalg.norm(g_emu)
    assert np.array_equal(net.loss_grad(r, t, 0.05)[1], grad)  # fixed order of all sums
    assert torch.equal(net.predict(r), net.predict(r, unfused=True))
    net.train_step(r, t, 0.05, 1e-3)
    d = net.params() - p
    live = np.abs(grad) > 1e-5
    assert np.allclose(d[live], -1e-3 * np.sign(grad[live]), rtol=1e-2)
    net.close()


def test_networks_that_share_an_output_buffer():
    """the output of one network's call, dropped by the caller, becomes the
    output of another's while nothing waits in between"""
    import torch
    from gimic_amd.surrogate import Network
    for seed in range(8):
        g = torch.Generator(device="cuda").manual_seed(seed)
        r = [12.0 * torch.rand((n, 3), generator=g, dtype=torch.float64, device="cuda") - 6.0
             for n in (100, 100)]
        nets = [Network(1.5, CS, np.linspace(0.5, 2.0, 9), seed=seed + k) for k in (0, 1)]
        torch.cuda.synchronize()
        print("case mlp shared output", seed, flush=True)
        nets[0].predict(r[0])
        nets[1].predict(r[1])
        got = nets[0].predict(r[0])
        torch.cuda.synchronize()
        assert torch.equal(got, nets[0].predict(r[0], unfused=True))
        for net in nets:
            net.close()


def test_batch_after_one_too_large_for_the_device():
    """a batch whose work buffers exceed the device's memory (22 TB; refused
    before any launch) is an error, and a batch within the earlier capacity
    then gets buffers again"""
    import ctypes
    import torch
    from gimic_amd import lib
    from gimic_amd.surrogate import Network
    g = torch.Generator(device="cuda").manual_seed(3)
    r = 12.0 * torch.rand((300, 3), generator=g, dtype=torch.float64, device="cuda") - 6.0
    t = torch.randn((300, 9), generator=g, dtype=torch.float64, device="cuda")
    net = Network(1.5, CS, np.linspace(0.5, 2.0, 9), seed=5)
    before = net.loss_grad(r, t, 0.05)
    print("case mlp batch of 2^36", flush=True)
    loss = ctypes.c_double()
    with pytest.raises(lib.GimicError, match="out of memory"):
        lib.check(net._lib.gimic_mlp_loss_grad(net._h, 1 << 36, ctypes.c_void_p(r.data_ptr()),
                                               ctypes.c_void_p(t.data_ptr()), 0.05,
                                               ctypes.byref(loss), None))
    after = net.loss_grad(r, t, 0.05)
    assert after[0] == before[0] and np.array_equal(after[1], before[1])
    net.close()
