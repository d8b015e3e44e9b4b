"""The shadow passes' tile drawing at its edges, bit for bit the oracle's brute-force restatement:
resolutions that end within a region, a tile and a lane's 2x2 texels, one wave per tile and four
(the calls with many tiles and with few), triangle lists shorter and longer than a wave's scan,
double-sided meshes (view depths of both signs), an empty list, and far planes and vertices that are not
finite."""
import dataclasses

import numpy as np
import pytest

import oracle as orc
from gpu_util import require_gpu
from stratusgfx_amd import _abi
from stratusgfx_amd import scene as sc
from stratusgfx_amd.gi import GiPass

pytestmark = pytest.mark.gpu


def _city(boxes, lights=4):
    s = sc.Scene(dataclasses.replace(sc.CITY_1080P, num_vpls=lights, num_city_boxes=boxes, city_half_extent=40.0))
    pos, col = s.triangles()
    return s, pos, col


def _atlases(layers, res, fmt, alloc):
    z, c = alloc((layers, 6, res, res), fmt), alloc((layers, 6, res, res), None)
    cz, cc = _abi.CubeAtlases(), _abi.CubeAtlases()
    for a, f, t in ((cz, fmt, z), (cc, _abi.TEXEL_RGBA8, c)):
        a.resolution, a.format, a.layers_per_atlas, a.num_atlases = res, f, layers, 1
        a.atlas[0] = t.ctypes.data if isinstance(t, np.ndarray) else t.data_ptr()
    return z, c, cz, cc


@pytest.mark.parametrize("res,lights,boxes,fmt,cull", [
    (1, 1, 30, _abi.TEXEL_F32, _abi.CULLING_CCW), (15, 3, 30, _abi.TEXEL_UNORM16, _abi.CULLING_NONE),
    (17, 2, 200, _abi.TEXEL_F16, _abi.CULLING_CW), (33, 2, 200, _abi.TEXEL_UNORM16, _abi.CULLING_CCW),
    (47, 2, 200, _abi.TEXEL_F32, _abi.CULLING_NONE), (194, 40, 60, _abi.TEXEL_F16, _abi.CULLING_CCW),
    (194, 40, 0, _abi.TEXEL_UNORM16, _abi.CULLING_CCW)])
def test_cubes(res, lights, boxes, fmt, cull):
    torch = require_gpu()
    s, pos, col = _city(max(boxes, 1), lights)
    if boxes == 0:
        pos, col = pos[:0], col[:0]
    vpls, _ = s.vpls()
    ent = np.stack([np.zeros(lights, np.int32), np.arange(lights, dtype=np.int32)], 1)
    kinds = {_abi.TEXEL_F32: torch.float32, _abi.TEXEL_F16: torch.float16, _abi.TEXEL_UNORM16: torch.int16,
             None: torch.int32}
    z, c, cz, cc = _atlases(lights, res, fmt, lambda sh, f: torch.full(sh, 3, dtype=kinds[f], device="cuda"))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    none = boxes == 0
    print(f"[tiles] cubes res {res} lights {lights} triangles {pos.shape[0]} fmt {fmt} cull {cull}", flush=True)
    GiPass(64, 64).render_vpl_cubes(None if none else d(pos), None if none else d(col.view(np.int32)), d(vpls),
                                    d(np.arange(lights, dtype=np.int32)), d(ent), cz, cc, cull=cull)
    torch.cuda.synchronize()
    hk = {_abi.TEXEL_F32: np.float32, _abi.TEXEL_F16: np.float16, _abi.TEXEL_UNORM16: np.uint16, None: np.uint32}
    hz, hc, hcz, hcc = _atlases(lights, res, fmt, lambda sh, f: np.zeros(sh, hk[f]))
    pick = np.array(sorted({0, lights // 2, lights - 1}), np.int32)
    orc.render_vpl_cubes(pos, col, vpls, pick, ent, _abi.REFERENCE_VPL_NEAR_PLANE, hcz, hcc, cull=cull)
    got, colour = z.cpu().numpy(), c.cpu().numpy().view(np.uint32)
    for u in pick:
        assert got[u].tobytes() == hz[u].tobytes(), f"distance of light {u}"
        assert np.array_equal(colour[u], hc[u]), f"colour of light {u}"


@pytest.mark.parametrize("res,boxes,cull", [(1, 30, _abi.CULLING_CCW), (31, 200, _abi.CULLING_NONE),
                                            (33, 200, _abi.CULLING_CW), (113, 200, _abi.CULLING_CCW),
                                            (1442, 8, _abi.CULLING_CCW), (50, 0, _abi.CULLING_CCW)])
def test_cascades(res, boxes, cull):
    torch = require_gpu()
    s, pos, _ = _city(max(boxes, 1))
    if boxes == 0:
        pos = pos[:0]
    csm = _abi.Csm()
    csm.resolution = res
    for k in range(4):
        for i in range(16):
            csm.cascadeProjViews[k][i] = s.csm.cascadeProjViews[k][i]
    depth = torch.full((4, res, res), -3.0, dtype=torch.float32, device="cuda")
    print(f"[tiles] cascades res {res} triangles {pos.shape[0]} cull {cull}", flush=True)
    GiPass(64, 64).render_csm(torch.from_numpy(pos).cuda() if boxes else None, csm, depth, cull=cull)
    torch.cuda.synchronize()
    want = orc.render_csm(pos, csm, slope=_abi.REFERENCE_CSM_SLOPE_FACTOR, cull=cull)
    assert np.array_equal(depth.cpu().numpy().view(np.uint32), want.view(np.uint32))


# lists within one scan and just beyond it, and either side of 3 triangles to 4 tiles
@pytest.mark.parametrize("res,lights,boxes", [(40, 2, 41), (40, 2, 42), (64, 8, 50), (64, 9, 50)])
def test_cubes_at_the_lines_between_the_forms(res, lights, boxes):
    test_cubes(res, lights, boxes, _abi.TEXEL_UNORM16, _abi.CULLING_NONE)


def _layers(n):
    """n large triangles one behind the other over +z and -x of the origin, wide in every tile of those faces."""
    pos = np.zeros((n, 3, 3), np.float32)
    for k in range(n):
        z = 2.0 + 0.5 * k
        pos[k] = [[-3 * z, -2 * z, z], [3 * z, -2 * z, z], [0.1 * k, 4 * z, z]]
        if k % 4 == 3:
            pos[k] = pos[k][:, [2, 1, 0]] * np.float32([-1, 1, 1])
    return pos, (np.arange(n, dtype=np.uint32) * 0x01030507 + 11)


# far: every triangle of a wave compares false with a NaN, which nothing is nearer than
@pytest.mark.parametrize("n,fmt", [(256, _abi.TEXEL_UNORM16), (256, _abi.TEXEL_F32), (300, _abi.TEXEL_UNORM16),
                                   (700, _abi.TEXEL_F32)])
@pytest.mark.parametrize("far,vertex", [(float("nan"), None), (float("inf"), None), (0.0, None), (-30.0, None),
                                        (120.0, float("nan")), (120.0, float("inf")), (120.0, -float("inf"))])
def test_cubes_not_finite(far, vertex, n, fmt):
    """Far planes that bound nothing and vertices that are nowhere, with n wide triangles in a tile: drawn by
    regions, by a wave a tile and by four."""
    torch = require_gpu()
    pos, col = _layers(n)
    if vertex is not None:
        pos[5, 1, 0] = pos[70, 2] = pos[200, 0, 2] = vertex
    vpls = np.zeros((3, _abi.VPL_FLOATS), np.float32)
    s, _, _ = _city(1, 3)
    vpls[:] = s.vpls()[0][:3]
    vpls[:, 0:3] = [[0, 0, 0], [0.3, -0.2, 0.1], [0, 0, 0]]
    vpls[:2, 13] = far
    vpls[2, 13] = 200.0  # a light beside them stays as it is
    ent = np.stack([np.zeros(3, np.int32), np.arange(3, dtype=np.int32)], 1)
    res, up = 32, np.arange(3, dtype=np.int32)
    kinds = {_abi.TEXEL_F32: torch.float32, _abi.TEXEL_UNORM16: torch.int16, None: torch.int32}
    z, c, cz, cc = _atlases(3, res, fmt, lambda sh, f: torch.full(sh, 3, dtype=kinds[f], device="cuda"))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    print(f"[tiles] cubes far {far} vertex {vertex} triangles {n} fmt {fmt}", flush=True)
    GiPass(64, 64).render_vpl_cubes(d(pos), d(col.view(np.int32)), d(vpls), d(up), d(ent), cz, cc,
                                    cull=_abi.CULLING_NONE)
    torch.cuda.synchronize()
    hk = {_abi.TEXEL_F32: np.float32, _abi.TEXEL_UNORM16: np.uint16, None: np.uint32}
    hz, hc, hcz, hcc = _atlases(3, res, fmt, lambda sh, f: np.zeros(sh, hk[f]))
    orc.render_vpl_cubes(pos, col, vpls, up, ent, _abi.REFERENCE_VPL_NEAR_PLANE, hcz, hcc, cull=_abi.CULLING_NONE)
    assert z.cpu().numpy().tobytes() == hz.tobytes()
    assert np.array_equal(c.cpu().numpy().view(np.uint32), hc)
    if not far > 0.0:  # the clears
        assert (hc[:2] == 0xFF000000).all()
    assert (hc[2] != 0xFF000000).any()


def test_every_light_of_a_call_in_batches():
    """24012 triangles: a call of 500 lights runs in several batches (48 B a triangle and light within 256 MB:
    232 lights).  Every light's cube is the one that a call of 50 lights, a single batch, gives it; those next
    to the boundaries are the oracle's."""
    torch = require_gpu()
    s = sc.Scene(dataclasses.replace(sc.CITY_1080P, num_vpls=500))
    pos, col = s.triangles()
    batch = (64 << 20) // (12 * ((pos.shape[0] + 3) // 4 * 4) + 6)
    assert pos.shape[0] == 24012 and batch == 232
    vpls, _ = s.vpls()
    ent = np.stack([np.arange(500) // 250, np.arange(500) % 250], 1).astype(np.int32)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731

    def atlases(alloc):  # 250 cubes in each of two
        z, c, cz, cc = _atlases(250, 16, _abi.TEXEL_UNORM16, lambda sh, f: alloc((2,) + sh, f))
        for a in (cz, cc):
            a.num_atlases = 2
            t = z if a is cz else c
            a.atlas[1] = t[1].ctypes.data if isinstance(t, np.ndarray) else t[1].data_ptr()
        return z, c, cz, cc

    dp, dc, dv, de, gi = d(pos), d(col.view(np.int32)), d(vpls), d(ent), GiPass(64, 64)
    got = []
    for step in (500, 50):
        z, c, cz, cc = atlases(lambda sh, f: torch.full(sh, 3, dtype=torch.int32 if f is None else torch.int16,
                                                        device="cuda"))
        print(f"[tiles] 500 lights, {step} a call", flush=True)
        for first in range(0, 500, step):
            gi.render_vpl_cubes(dp, dc, dv, d(np.arange(first, first + step, dtype=np.int32)), de, cz, cc)
        torch.cuda.synchronize()
        got.append([t.view(500, 6, 16, 16).cpu().numpy() for t in (z, c)])
    for one, few in zip(*got):
        assert np.array_equal(one, few), np.nonzero((one != few).any(axis=(1, 2, 3)))[0]
    hz, hc, hcz, hcc = atlases(lambda sh, f: np.zeros(sh, np.uint32 if f is None else np.uint16))
    pick = np.array([batch - 1, batch, 2 * batch - 1, 2 * batch, 499], np.int32)
    orc.render_vpl_cubes(pos, col, vpls, pick, ent, _abi.REFERENCE_VPL_NEAR_PLANE, hcz, hcc)
    z, c = got[0]
    for u in pick:
        assert z[u].tobytes() == hz.reshape(500, 6, 16, 16)[u].tobytes(), f"distance of light {u}"
        assert np.array_equal(c.view(np.uint32)[u], hc.reshape(500, 6, 16, 16)[u]), f"colour of light {u}"


# meshes of one to 256 triangles, drawn by regions: 16 and 17 in one (in their order, and near ones first),
# sides that cut a region and a lane's 2x2 texels
@pytest.mark.parametrize("n,res,fmt,cull", [
    (1, 32, _abi.TEXEL_F32, _abi.CULLING_NONE), (16, 31, _abi.TEXEL_F16, _abi.CULLING_NONE),
    (17, 33, _abi.TEXEL_UNORM16, _abi.CULLING_NONE), (64, 1, _abi.TEXEL_F32, _abi.CULLING_CCW),
    (65, 47, _abi.TEXEL_F32, _abi.CULLING_CW), (255, 64, _abi.TEXEL_F16, _abi.CULLING_NONE),
    (256, 47, _abi.TEXEL_UNORM16, _abi.CULLING_NONE), (257, 47, _abi.TEXEL_UNORM16, _abi.CULLING_NONE)])
@pytest.mark.parametrize("kind", ["layers", "ties", "city"])
def test_cubes_of_few_triangles(n, res, fmt, cull, kind):
    """Layers over each other from near to far and back, the same triangle n times and within a step of each
    format (the first of equal keys stays), and a part of a city: the oracle's bits."""
    torch = require_gpu()
    rng = np.random.default_rng(n)
    s, pos, col = _city(30, 3)
    vpls = s.vpls()[0][:3].copy()
    if kind == "city":
        pos, col = pos[:n], col[:n]
    else:
        pos, col = _layers(n)
        if kind == "ties":
            pos = np.repeat(pos[:1], n, 0)
            pos[n // 2:] *= np.float32(1.0) + (rng.integers(-6, 7, (n - n // 2, 1, 1)) * 2.0 ** -18).astype(np.float32)
        pos = np.ascontiguousarray(pos[rng.permutation(n)])
        vpls[:, 0:3] = [[0, 0, 0], [0.3, -0.2, 0.1], [-0.5, 0.4, -1.0]]
        vpls[:, 13] = [100.0, 300.0, 40.0]
    col = (np.arange(n, dtype=np.uint32) * 0x010307 + 5)  # every triangle its own
    ent = np.stack([np.zeros(3, np.int32), np.arange(3, dtype=np.int32)], 1)
    kinds = {_abi.TEXEL_F32: torch.float32, _abi.TEXEL_F16: torch.float16, _abi.TEXEL_UNORM16: torch.int16,
             None: torch.int32}
    z, c, cz, cc = _atlases(3, res, fmt, lambda sh, f: torch.full(sh, 3, dtype=kinds[f], device="cuda"))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    print(f"[tiles] cubes of {n} triangles ({kind}) res {res} fmt {fmt} cull {cull}", flush=True)
    up = np.arange(3, dtype=np.int32)
    GiPass(64, 64).render_vpl_cubes(d(pos), d(col.view(np.int32)), d(vpls), d(up), d(ent), cz, cc, cull=cull)
    torch.cuda.synchronize()
    hk = {_abi.TEXEL_F32: np.float32, _abi.TEXEL_F16: np.float16, _abi.TEXEL_UNORM16: np.uint16, None: np.uint32}
    hz, hc, hcz, hcc = _atlases(3, res, fmt, lambda sh, f: np.zeros(sh, hk[f]))
    orc.render_vpl_cubes(pos, col, vpls, up, ent, _abi.REFERENCE_VPL_NEAR_PLANE, hcz, hcc, cull=cull)
    assert z.cpu().numpy().tobytes() == hz.tobytes()
    assert np.array_equal(c.cpu().numpy().view(np.uint32), hc)
