"""The network's kernels where their tiles are cut: images of one tile, a pixel more or less, odd sides
(the pooling's last row and column) and a single row, against the oracle; the fused network of the frame
path against the training path's separate kernels, bit for bit."""
import numpy as np
import pytest

import kpcn_check
import kpcn_oracle as ko
from gpu_util import Case, require_gpu, small
from stratusgfx_amd import _abi, kpcn
from stratusgfx_amd import scene as sc
from stratusgfx_amd.gi import GiPass

pytestmark = pytest.mark.gpu

SIZES = [(16, 16), (15, 17), (33, 31), (1, 70)]


def _bf(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda().to(torch.bfloat16)


@pytest.mark.parametrize("H,W", SIZES)
def test_convolution_and_weight_gradient(H, W):
    torch = require_gpu()
    lib = _abi.load()
    rng = np.random.default_rng(H * W)
    Wt = ko.to_bf16(rng.normal(0, 0.1, (9, 32, 32)))
    b = rng.normal(0, 0.1, 32).astype(np.float32)
    x, dy = (ko.to_bf16(rng.normal(0, 1, (H, W, 32))) for _ in range(2))
    xd, dyd, wd, bd = _bf(torch, x), _bf(torch, dy), _bf(torch, Wt), torch.from_numpy(b).cuda()
    want = ko.conv3x3(x, Wt, b.astype(np.float64))
    for f32 in (0, 1):
        out = torch.full((H + 1, W, 32), 7.0, dtype=torch.float32 if f32 else torch.bfloat16, device="cuda")
        _abi.call(lib, "sgi_kpcn_conv3x3", xd.data_ptr(), 0, wd.data_ptr(), bd.data_ptr(), 0, H, W, out.data_ptr(),
                  f32, 0)
        torch.cuda.synchronize()
        got = out.float().cpu().numpy().astype(np.float64)
        assert (got[H] == 7.0).all()
        tol = 1e-5 * np.abs(want).max() if f32 else 2.0 ** -7 * np.abs(want) + 1e-6
        assert (np.abs(got[:H] - (want if f32 else ko.to_bf16(want))) <= tol).all()
    parts = torch.empty(int(lib.sgi_kpcn_wgrad_partials(H, W)), dtype=torch.float32, device="cuda")
    grad = torch.empty(ko.LAYER_PARAMS, dtype=torch.float32, device="cuda")
    _abi.call(lib, "sgi_kpcn_conv3x3_wgrad", xd.data_ptr(), dyd.data_ptr(), 0, H, W, parts.data_ptr(),
              grad.data_ptr(), 0)
    torch.cuda.synchronize()
    dW, db, _ = ko.conv3x3_backward(x, dy, np.zeros((9, 32, 32)))
    g, want_g = grad.cpu().numpy().astype(np.float64), np.concatenate([dW.reshape(-1), db])
    assert np.linalg.norm(g - want_g) / np.linalg.norm(want_g) <= 1e-5


# (the coarsest level has more than one pixel: over one the filter has no gradient and the check no scale)
@pytest.mark.parametrize("H,W", [(48, 32), (33, 31), (50, 67)])
def test_training_step(H, W):
    torch = require_gpu()
    rng = np.random.default_rng(H + W)
    params = kpcn.init_params(7)
    feat = np.zeros((H, W, 32))
    feat[..., :10] = rng.normal(0, 1, (H, W, 10))
    feat = ko.to_bf16(feat)
    rad = rng.uniform(0, 2, (H, W, 3)).astype(np.float32)
    target = rng.uniform(0.1, 1.5, (H, W, 3)).astype(np.float32)
    tr = kpcn.Trainer(kpcn.Weights(params), H, W)
    tr.zero_grad()
    fd, rd, td = _bf(torch, feat), torch.from_numpy(rad).cuda(), torch.from_numpy(target).cuda()
    tr.forward(fd, rd)
    tr.loss_backward(td, err_weight=0.1)
    torch.cuda.synchronize()
    kpcn_check.compare(tr, params, feat, rad, target, 0.1)


@pytest.mark.parametrize("H,W", SIZES + [(50, 67)])
def test_fused_network_is_the_training_path(H, W):
    torch = require_gpu()
    case = Case(small(sc.CORNELL_640x360, name=f"cornell-{W}x{H}-8vpl", width=W, height=H, num_vpls=8, cube_res=16,
                      csm_res=64))
    gi = GiPass(W, H, 16, 12)
    gi.set_frame(case.dev.frame)
    gi.set_csm(case.dev.csm_struct())
    rng = np.random.default_rng(W)
    f32 = dict(dtype=torch.float32, device="cuda")
    lit, col, res = (torch.from_numpy(rng.uniform(0.1, 2, (H, W, c)).astype(np.float32)).cuda() for c in (3, 3, 4))
    vis = torch.tensor([8], dtype=torch.int32, device="cuda")
    wts = kpcn.Weights(kpcn.init_params(3))
    outs = [torch.zeros((H, W, c), **f32) for c in (3, 3, 4)]
    g = case.dev.gbuffer()
    gi.denoise_learned(g, None, vis, lit, col, res, None, None, wts.net(), float("inf"), gi.kpcn_workspace(), *outs,
                       torch.zeros((H, W), **f32))
    feat, rad = torch.empty((H, W, 32), dtype=torch.bfloat16, device="cuda"), torch.empty((H, W, 3), **f32)
    gi.kpcn_features(g, res, feat, rad)
    want = kpcn.Trainer(wts, H, W).forward(feat, rad)
    torch.cuda.synchronize()
    assert torch.equal(outs[2][..., :3], want)


def test_gradients_of_samples_add():
    """Two samples without zero_grad between them leave the sum of their gradients: one addition a parameter."""
    torch = require_gpu()
    H, W = 40, 56
    rng = np.random.default_rng(9)
    tr = kpcn.Trainer(kpcn.Weights(kpcn.init_params(7)), H, W)
    samples = []
    for _ in range(2):
        feat = np.zeros((H, W, 32))
        feat[..., :10] = rng.normal(0, 1, (H, W, 10))
        rad, target = (torch.from_numpy(rng.uniform(0.1, 2, (H, W, 3)).astype(np.float32)).cuda() for _ in range(2))
        samples.append((_bf(torch, feat), rad, target))

    def run(which):
        tr.zero_grad()
        for feat, rad, target in which:
            tr.forward(feat, rad)
            tr.loss_backward(target, err_weight=0.1)
        torch.cuda.synchronize()
        return tr.grad.clone()

    first, second = run(samples[:1]), run(samples[1:])
    assert not torch.equal(first, second) and bool((first != 0).any()) and bool((second != 0).any())
    assert torch.equal(run(samples), first + second)
