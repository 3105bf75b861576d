"""Tables of directions that are no pinhole's: the renderer takes the traversals
made for them, and every traversal, the block form called directly among them,
gives the same images.  The block form against the oracle."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _scene(pkg, gpu, n):
    model = pkg.SimModelDO([pkg.scenes.solid("ellipsoid", 900, seed=5), pkg.scenes.solid("box", 3000, seed=6)],
                           [i % 2 for i in range(n)], device=gpu)
    pkg.SimBVH(gpu, model)
    return model


def _fisheye(ren):
    d, R = ren.dirs[:, :3].clone(), 2 * ren.width
    c = d[0] + d[R - 1] + d[-1] + d[-R]
    c = c / c.norm()
    th = torch.acos((d * c).sum(1).clamp(-1, 1))
    perp = d - (d * c).sum(1, keepdim=True) * c
    perp = perp / perp.norm(dim=1, keepdim=True).clamp_min(1e-9)
    a = 0.9 * torch.tan(th)
    ren.dirs[:, :3] = torch.cos(a)[:, None] * c + torch.sin(a)[:, None] * perp


@pytest.mark.parametrize("n,res,expect", [(2, 64, 1), (3, 132, 1), (600, 64, 1), (128, 128, 2)])
def test_other_tables_take_other_traversals(pkg, gpu, n, res, expect):
    model = _scene(pkg, gpu, n)
    ren = pkg.RaycastRendererDO(gpu, model, cameraPos=(0.0, 1.6, 5.5), resolution=res)
    ren.lookAt((0.0, 0.45, 0.0))
    assert ren._traversal(n) == 0
    _fisheye(ren)
    assert ren._traversal(n) == expect
    img = ren.render_depth().clone()
    assert int((img > 0).sum()) > 0
    for t in (0, 1, 2):                     # each form called directly
        cam = pkg._lib.Camera()
        C.pointer(cam)[0] = ren.camera
        cam.traversal = t
        pkg.lib.ffsrl_render(model.batch, cam, 0, n, ren.depth.data_ptr(), None, None, None, None, None, None,
                             model.stream())
        assert torch.equal(img.view(torch.int32), ren.depth.view(torch.int32)), t
    ren.set_traversal(2)
    assert ren._traversal(n) == 2           # a chosen form is kept
    ren.set_traversal(0)
    ren.lookAt((0.0, 0.45, 0.0))            # a table of its own again
    assert ren._traversal(n) == 0
    with torch.inference_mode():
        assert pkg.RaycastRendererDO(gpu, model, resolution=64)._traversal(n) == 0


@pytest.mark.parametrize("res", [20, 128])
def test_block_form_equals_the_oracle(pkg, orc, gpu, res):
    mesh = pkg.scenes.solid("ellipsoid", 3000, seed=7)
    model = pkg.SimModelDO([mesh], [0], device=gpu)
    pkg.SimBVH(gpu, model)
    ren = pkg.RaycastRendererDO(gpu, model, cameraPos=(0.0, 1.6, 5.5), resolution=res)
    ren.lookAt((0.0, 0.45, 0.0))
    hit = torch.full((4 * res * res,), -7, dtype=torch.int32, device=gpu)
    thit = torch.zeros(4 * res * res, dtype=torch.float32, device=gpu)
    depth = ren.render_depth(hit=hit, thit=thit)
    torch.cuda.synchronize()
    t, x = model.topo[0], model.vertex().cpu().numpy()
    bvh = {"left": t.left, "first": t.first, "count": t.count, "level": t.level, "tri_map": t.tri_map}
    mn, mx = orc.refit(bvh, mesh.tris, x)
    d, h, tt, _ = orc.render_depth(res, res, np.asarray(ren.camera.origin[:], np.float32), ren.dirs.cpu().numpy(), bvh,
                                   mn, mx, mesh.tris, x)
    assert (h >= 0).sum() > 0 and np.array_equal(hit.cpu().numpy(), h)
    assert np.array_equal(thit.cpu().numpy(), tt) and np.array_equal(depth[0].cpu().numpy(), d)


@pytest.mark.parametrize("n", [2, 64])
def test_block_form_on_odd_tables_and_values(pkg, gpu, n):
    """The block form called directly where the renderer would not choose it."""
    model = _scene(pkg, gpu, n)
    bvh = pkg.SimBVH(gpu, model)
    ren = pkg.RaycastRendererDO(gpu, model, cameraPos=(0.0, 1.6, 5.5), resolution=132)
    ren.lookAt((0.0, 0.45, 0.0))
    keep = ren.dirs.clone()
    g = torch.Generator(device=gpu)
    g.manual_seed(1)

    def compare():
        got = []
        for t in (1, 0):
            ren.set_traversal(t)
            hit = torch.full((n, 4 * 132 * 132), -7, dtype=torch.int32, device=gpu)
            thit = torch.full((n, 4 * 132 * 132), -7.0, device=gpu)
            pkg.lib.ffsrl_render(model.batch, ren.camera, 0, n, ren.depth.data_ptr(), None, None, None, None,
                                 hit.data_ptr(), thit.data_ptr(), model.stream())
            got.append((hit, thit.view(torch.int32), ren.depth.clone().view(torch.int32)))
        assert all(torch.equal(a, b) for a, b in zip(*got)) and int((got[0][0] >= 0).sum()) > 0

    for table in (keep[torch.randperm(keep.shape[0], generator=g, device=gpu)],
                  torch.cat([keep[:5000], keep[5000:9000] * 1.5, keep[9000:]])):
        ren.dirs.copy_(table)
        compare()
    ren.dirs.copy_(keep)
    for k, bad in enumerate((float("nan"), float("inf"), 3e38)):
        model.x[int(model.env_vbase[k % n]) + 7 * k + 50, k % 3] = bad
    compare()                               # bounds older than the positions
    bvh.refitBVH()
    compare()
