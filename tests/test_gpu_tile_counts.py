"""Frames of 1, 127, 128, 129 and 8 x 17 tiles of 16 x 16: the blocks of the gathers, tile culling and
direct light are dealt to the XCDs in chunks of 16 tiles, so a launch holds up to 127 blocks without a
tile.  Every tile has to be done once, and nothing written beyond the last one.  The cubes are of even, odd and
unit size: a lookup near a texel's edge takes the exact formula, any other an estimate."""
import numpy as np
import pytest

import oracle as orc
from gpu_util import Case, assert_tiles_equal, require_gpu, small
from stratusgfx_amd import _abi
from stratusgfx_amd import scene as sc
from stratusgfx_amd.gi import GiPass

pytestmark = pytest.mark.gpu

REL_L2 = 1e-4  # FP32 images, the bound of every parity test


@pytest.mark.parametrize("W,H,cube", [(16, 16, 1), (2032, 16, 32), (1024, 32, 31), (2049, 7, 32), (125, 270, 7)])
def test_every_tile_once(W, H, cube):
    torch = require_gpu()
    case = Case(small(sc.CORNELL_640x360, name=f"cornell-{W}x{H}-24vpl", width=W, height=H, num_vpls=24,
                      cube_res=cube, csm_res=256))
    ts, K = 16, 7
    gi = GiPass(W, H, ts, K)
    gi.set_frame(case.dev.frame)
    gi.set_csm(case.dev.csm_struct())
    upd, vis, ent = case.oracle_cull()
    d_upd, d_vis = torch.from_numpy(upd).cuda(), torch.from_numpy(vis).cuda()
    d_ent = torch.from_numpy(np.ascontiguousarray(ent)).cuda()
    g = case.dev.gbuffer()

    def images():  # the frame's rows and one row more, which stays as it is
        return [torch.full((H + 1, W, c), 7.0, dtype=torch.float32, device="cuda") for c in (3, 4)]

    def check(got, want):
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert orc.rel_l2(a[:H].cpu().numpy(), b) <= REL_L2
            assert bool((a[H] == 7.0).all())

    _, o_tiles = orc.cull_tiles(case.host.frame, case.hg, ts, K, upd, vis)
    tiles = torch.full((gi.num_tiles + 1, 1 + K), -5, dtype=torch.int32, device="cuda")
    gi.cull_tiles(g, d_upd, d_vis, tiles[:gi.num_tiles])
    torch.cuda.synchronize()
    assert_tiles_equal(tiles[:gi.num_tiles].cpu().numpy(), o_tiles)
    assert bool((tiles[gi.num_tiles] == -5).all())

    args = (case.host.frame, case.hg, upd, int(vis[0]), ent, case.hcubes)
    col, res = images()
    gi.gather(g, d_upd, d_vis, d_ent, case.dev.cubes(), tiles[:gi.num_tiles], col[:H], res[:H])
    check((col, res), orc.gather(*args, tiles=o_tiles, tile_size=ts, K=K, mode=orc.GATHER_TILES))
    col, res = images()
    gi.gather(g, d_upd, d_vis, d_ent, case.dev.cubes(), None, col[:H], res[:H])
    check((col, res), orc.gather(*args, mode=orc.GATHER_RANDOM))
    for mode, omode, kw in ((_abi.GATHER_ALL, orc.GATHER_CONVERGED, {}),
                            (_abi.GATHER_SAMPLES, orc.GATHER_SAMPLES, dict(samples=4, rejection_limit=5))):
        col, res = images()
        gi.gather_ex(g, d_upd, d_vis, d_ent, case.dev.cubes(), None, col[:H], res[:H], mode=mode, **kw)
        check((col, res), orc.gather(*args, mode=omode, precision=0, **kw))
    lit = images()[0]
    gi.direct_light(g, lit[:H])
    check((lit,), (orc.direct_light(case.host.frame, case.hcsm, case.hg),))


@pytest.mark.parametrize("radius", [None, 0.5, 6.0, 1.0e6])
@pytest.mark.parametrize("accumulate_fp64", [False, True])
def test_converged_drops_only_rejected(radius, accumulate_fp64):
    """The converged gather drops a VPL for a whole wave where none of its pixels can accept it: radii as
    generated, small enough to drop nearly all, about a tile's extent, and without end."""
    torch = require_gpu()
    W, H = 200, 75
    case = Case(small(sc.CORNELL_640x360, name="cornell-200x75-90vpl", width=W, height=H, num_vpls=90, cube_res=16,
                      csm_res=64))
    gi = GiPass(W, H, 16, 12)
    gi.set_frame(case.dev.frame)
    gi.set_csm(case.dev.csm_struct())
    upd, vis, ent = case.oracle_cull()
    if radius is not None:
        upd = upd.copy()
        upd[:, 12] = radius
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    col = torch.zeros((H, W, 3), dtype=torch.float32, device="cuda")
    res = torch.zeros((H, W, 4), dtype=torch.float32, device="cuda")
    gi.gather_ex(case.dev.gbuffer(), d(upd), d(vis), d(ent), case.dev.cubes(), None, col, res, mode=_abi.GATHER_ALL,
                 accumulate_fp64=accumulate_fp64)
    torch.cuda.synchronize()
    oc, orr = orc.gather(case.host.frame, case.hg, upd, int(vis[0]), ent, case.hcubes, mode=orc.GATHER_CONVERGED,
                         precision=0)
    assert orc.rel_l2(res.cpu().numpy(), orr) <= REL_L2
    assert float(np.abs(res[..., 3].cpu().numpy().astype(np.float64) - orr[..., 3]).max()) < 1e-3
    assert orc.rel_l2(col.cpu().numpy(), oc) <= REL_L2


@pytest.fixture(scope="module")
def city():
    return Case(small(sc.CITY_1080P, name="city-200x120-1500vpl", width=200, height=120, num_vpls=1500, cube_res=8,
                      csm_res=256))


@pytest.mark.parametrize("radius", [None, -40.0, 0.0, 60.0, 1.0e6, float("nan")])
@pytest.mark.parametrize("ts,K", [(8, 64), (16, 64), (16, 12), (32, 64)])
def test_tile_lists_by_rank(city, ts, K, radius):
    """Tile lists formed by counting smaller keys, against the oracle bit for bit: as generated, radii that
    leave more candidates than there are keys, none, or negative ratios (the insertions run instead)."""
    torch = require_gpu()
    gi = GiPass(city.w.width, city.w.height, ts, K)
    gi.set_frame(city.dev.frame)
    gi.set_csm(city.dev.csm_struct())
    upd, vis, _ = city.oracle_cull()
    if radius is not None:
        upd = upd.copy()
        upd[:, 12] = radius
    _, want = orc.cull_tiles(city.host.frame, city.hg, ts, K, upd, vis)
    tiles = torch.full((gi.num_tiles, 1 + K), -5, dtype=torch.int32, device="cuda")
    gi.cull_tiles(city.dev.gbuffer(), torch.from_numpy(upd).cuda(), torch.from_numpy(vis).cuda(), tiles)
    torch.cuda.synchronize()
    assert_tiles_equal(tiles.cpu().numpy(), want)
