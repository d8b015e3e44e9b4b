"""FXAA on both of its tile sizes (32 x 32 below 4 M pixels, 64 x 64 above), at frame edges that cut a tile
and where walks leave the halo, and the TAA history off 16-byte alignment: the oracle's bytes."""
import numpy as np
import pytest

import oracle as orc
from gpu_util import require_gpu
from stratusgfx_amd.gi import GiPass

pytestmark = pytest.mark.gpu


def _image(H, W, seed):
    """Long edges with slight steps (walks of full length), blocks and noise."""
    rng = np.random.default_rng(seed)
    base = np.kron(rng.integers(0, 256, (H // 11 + 1, W // 37 + 1, 3)), np.ones((11, 37, 1)))[:H, :W]
    base[:, W // 2:] = base[:1, W // 2:] // 2 + (np.arange(H) * 3 % 128)[:, None, None] // 8
    noisy = rng.random((H, W, 1)) < 0.02
    t = np.where(noisy, rng.integers(0, 256, (H, W, 3)), base).astype(np.uint32)
    return t[..., 0] | t[..., 1] << 8 | t[..., 2] << 16 | np.uint32(255 << 24)


@pytest.mark.parametrize("H,W", [(1, 1), (31, 33), (32, 64), (97, 250), (2051, 2049)])
def test_fxaa(H, W):
    torch = require_gpu()
    img = _image(H, W, H + W)
    gi = GiPass(W, H, 16, 12)
    out = torch.full((H + 1, W), 5, dtype=torch.int32, device="cuda")
    gi.fxaa(torch.from_numpy(img.view(np.int32)).cuda(), out[:H])
    torch.cuda.synchronize()
    assert np.array_equal(out[:H].cpu().numpy().view(np.uint32), orc.fxaa(img)[1])
    assert bool((out[H] == 5).all())


@pytest.mark.parametrize("shift", [0, 1, 2])
def test_taa_history_alignment(shift):
    torch = require_gpu()
    H, W = 7, 13  # 273 values: one is left after the fours
    rng = np.random.default_rng(shift)
    v = rng.uniform(-0.5, 2.0, (H, W, 3)).astype(np.float32)
    buf = torch.zeros(2, H * W * 3 + 4, dtype=torch.float32, device="cuda")
    src, dst = (b[shift:shift + v.size].view(H, W, 3) for b in buf)
    src.copy_(torch.from_numpy(v))
    GiPass(W, H, 16, 12).taa_history(src, dst)
    torch.cuda.synchronize()
    assert np.array_equal(dst.cpu().numpy().view(np.uint32), orc.taa_history(v).view(np.uint32))
    assert bool((buf[1, :shift] == 0).all()) and bool((buf[1, shift + v.size:] == 0).all())


@pytest.mark.parametrize("H,W", [(1, 1), (2, 3), (4, 4), (11, 31), (1, 342), (1, 343), (19, 18)])
def test_taa_history_remainders(H, W):
    """One to three values after the fours, and none, at and beside a block's 1024."""
    torch = require_gpu()
    v = np.random.default_rng(W).uniform(-0.5, 2.0, (H, W, 3)).astype(np.float32)
    v.reshape(-1)[:3] = [np.nan, np.inf, -np.inf]
    dst = torch.full((v.size + 4,), -3.0, dtype=torch.float32, device="cuda")
    GiPass(W, H, 16, 12).taa_history(torch.from_numpy(v).cuda(), dst[:v.size].view(H, W, 3))
    torch.cuda.synchronize()
    assert np.array_equal(dst[:v.size].cpu().numpy().view(np.uint32), orc.taa_history(v).view(np.uint32).reshape(-1))
    assert bool((dst[v.size:] == -3.0).all())
