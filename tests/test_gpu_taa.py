"""sgi_taa (taa.fs) on the GPU: bit for bit the oracle's restatement on random
frames, histories and velocities (some reaching past the edges, where the
bilinear history taps clamp), and without a velocity plane; an output that
aliases an input is refused."""
import numpy as np
import pytest

import oracle as orc
from gpu_util import require_gpu
from stratusgfx_amd import _abi
from stratusgfx_amd.gi import GiPass

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("with_velocity", [True, False])
def test_taa_bit_exact(with_velocity):
    torch = require_gpu()
    H, W = 97, 203
    rng = np.random.default_rng(5)
    cur = np.exp(rng.uniform(-6, 3, (H, W, 3))).astype(np.float32)
    hist = np.exp(rng.uniform(-6, 3, (H, W, 3))).astype(np.float32)
    vel = (rng.standard_normal((H, W, 2)) * 0.02).astype(np.float32) if with_velocity else None
    gi = GiPass(W, H, 16, 12)
    d = lambda a: None if a is None else torch.from_numpy(a).cuda()  # noqa: E731
    out = torch.zeros((H, W, 3), dtype=torch.float32, device="cuda")
    gi.taa(d(cur), d(hist), d(vel), out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    want = orc.taa(cur, hist, vel)
    bad = got.view(np.uint32) != want.view(np.uint32)
    print(f"[taa] {W}x{H} velocity={with_velocity}: {int(bad.sum())} of {bad.size} values differ; "
          f"max rel {float(np.max(np.abs(got - want) / np.maximum(np.abs(want), 1e-30))):.2e}", flush=True)
    assert not bad.any()
    with pytest.raises(_abi.SgiError):
        gi.taa(out, d(hist), None, out)


@pytest.mark.parametrize("H,W", [(256, 768), (640, 768)])  # the two forms of the clamp
def test_taa_clamp_near_ties(H, W):
    """Histories within a few ulp of the neighbourhood's least and largest values, which lie a few ulp apart
    or are equal: the tone curve rounds, so that neighbours may come out the wrong way round, and the clamp
    has to choose as the curve's values do.  From 1e-6 to where the curve is 1."""
    torch = require_gpu()
    rng = np.random.default_rng(11)
    cur = np.kron(np.exp(rng.uniform(-14, 8, (H // 4, W // 4, 3))), np.ones((4, 4, 1))).astype(np.float32)
    cur[:8, :8], cur[:8, 8:16], cur[:8, 16:24], cur[:8, 24:32] = 0.0, 1e16, 3e7, 1e-30
    bits = cur.view(np.int32)
    spread = rng.integers(0, 4, (H // 4, W // 4, 1)).repeat(4, 0).repeat(4, 1)  # 0: all equal
    near = (bits + rng.integers(-3, 4, bits.shape) * spread).clip(0)
    cur = near.astype(np.int32).view(np.float32)
    step = rng.choice([1, 2, 8, 40, 1000], (H, W, 1)) * rng.integers(-2, 3, bits.shape)
    hist = np.ascontiguousarray((cur.view(np.int32) + step).clip(0).astype(np.int32).view(np.float32))
    gi = GiPass(W, H, 16, 12)
    out = torch.zeros((H, W, 3), dtype=torch.float32, device="cuda")
    gi.taa(torch.from_numpy(cur).cuda(), torch.from_numpy(hist).cuda(), None, out)
    torch.cuda.synchronize()
    got, want = out.cpu().numpy(), orc.taa(cur, hist, None)
    bad = (got.view(np.uint32) != want.view(np.uint32)) & ~(np.isnan(got) & np.isnan(want))
    print(f"[taa] near ties: {int(bad.sum())} of {bad.size} values differ", flush=True)
    assert not bad.any()
