"""The a-trous filter at the edges of its regions, in its three forms: one pixel per thread below 750 blocks
of 64 x 4 pixels, a column of two below 1800 and of four from there on, whose pixels lie a lattice step
(2, 4, 8) apart in regions of 64 x 16 and 64 x 32.  Pixels past the frame's last row or column have to
stay unwritten."""
import numpy as np
import pytest

import oracle as orc
from gpu_util import Case, require_gpu, small
from stratusgfx_amd import scene as sc
from stratusgfx_amd.gi import GiPass

pytestmark = pytest.mark.gpu

REL_L2 = 1e-4  # FP32 images, the bound of every parity test


@pytest.mark.parametrize("W,H", [(1, 1), (3, 33), (64, 32), (65, 31), (63, 40), (130, 70), (517, 375), (64, 3203), (2049, 97),
                                 (517, 803), (64, 7201), (2049, 221)])
def test_denoise_matches_oracle(W, H):
    torch = require_gpu()
    case = Case(small(sc.CORNELL_640x360, name=f"cornell-{W}x{H}-12vpl", width=W, height=H, num_vpls=12,
                      cube_res=16, csm_res=128))
    gi = GiPass(W, H, 16, 12)
    gi.set_frame(case.dev.frame)
    gi.set_csm(case.dev.csm_struct())
    rng = np.random.default_rng(W + H)
    lit, col = (rng.random((H, W, 3), dtype=np.float32) for _ in range(2))
    res = np.exp(rng.uniform(-3, 3, (H, W, 4))).astype(np.float32)
    vis = np.array([12], np.int32)
    want = orc.denoise(case.host.frame, case.hg, None, 12, lit, col, res)
    t = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    got = [torch.full((H + 1, W, c), 7.0, dtype=torch.float32, device="cuda") for c in (3, 3, 4, 1)]
    gi.denoise(case.dev.gbuffer(), None, t(vis), t(lit), t(col), t(res), None, None, *[o[:H] for o in got])
    torch.cuda.synchronize()
    for name, o, w in zip(("combined", "gi", "reservoir", "history"), got, want):
        assert bool((o[H] == 7.0).all()), name
        assert orc.rel_l2(o[:H].cpu().numpy().reshape(w.shape), w) <= REL_L2, name
