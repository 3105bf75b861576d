"""The automatic (block) traversal gives the hits, distances and images of the
one-ray-per-lane traversal bit for bit, for every block size, image edges that
cut blocks, cameras outside, inside and far away, rays with zero components,
tables of directions that are no pinhole's, leaves of several triangles, list
overflow, bounds older than the positions, and positions that are not finite."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CAMERAS = [((0.0, 1.6, 5.5), (0.0, 0.45, 0.0), 19.2, 19.2), ((0.1, 0.5, 0.05), (1.0, 0.6, 0.3), 80.0, 50.0),
           ((0.0, 0.45, 3.0), (0.0, 0.45, 0.0), 19.2, 24.0), ((10.0, 40.0, 60.0), (0.0, 0.4, 0.0), 2.0, 2.0)]


def _model(pkg, gpu, scene, n):
    sc = pkg.scenes
    if scene == "liver":
        us = importlib.import_module("ff-srl_amd.usd_scene")
        return pkg.SimModelDO([us.merged_mesh(us.scene("tests/golden/liver_retraction.npz"))], [0] * n, device=gpu)
    if scene == "cube":  # planar faces, vertices in the camera's planes
        return pkg.SimModelDO([sc.cube_grid(7)], [0] * n, device=gpu)
    meshes = [sc.solid("ellipsoid" if i % 2 else "box", t, seed=i) for i, t in enumerate((900, 6000, 30000))]
    return pkg.SimModelDO(meshes, [i % 3 for i in range(n)], device=gpu)


def _compare(pkg, gpu, model, ren, rgb=False):
    n, res = model.numEnvs, ren.height
    got = []
    for traversal in (1, 0):
        ren.set_traversal(traversal)
        hit = torch.full((n, 4 * res * res), -7, dtype=torch.int32, device=gpu)
        thit = torch.full((n, 4 * res * res), -7.0, device=gpu)
        got.append([hit, thit, ren.render_depth(hit=hit, thit=thit).clone()])
        if rgb:
            pix, dep = ren.render_rgbd()
            got[-1] += [pix.clone(), dep.clone()]
    for a, b in zip(*got):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    return int((got[0][0] >= 0).sum())


@pytest.mark.parametrize("scene", ["solids", "cube", "liver"])
@pytest.mark.parametrize("n,res", [(1, 4), (2, 20), (3, 132), (24, 132), (64, 132)])  # 1x1, 2x1 and 2x2 blocks
def test_block_equals_per_ray(pkg, gpu, scene, n, res):
    model = _model(pkg, gpu, scene, n)
    big = 8.0 if scene == "liver" else 1.0
    g = torch.Generator(device=gpu)
    g.manual_seed(n)
    if scene != "cube":
        model.x[:, :3] += 0.02 * big * torch.randn((model.numVertices, 3), generator=g, device=gpu)
    pkg.SimBVH(gpu, model)
    hits = 0
    for pos, at, ha, va in CAMERAS[:4 if n < 24 else 1]:
        at = (0.0, 8.0, 0.0) if scene == "liver" else at
        ren = pkg.RaycastRendererDO(gpu, model, cameraPos=[big * c for c in pos], resolution=res,
                                    horizontalAperture=ha, verticalAperture=va,
                                    render_mode=pkg.RenderMode.vertex_color)
        ren.lookAt(at)
        hits += _compare(pkg, gpu, model, ren, rgb=True)
    assert hits > 0


@pytest.mark.parametrize("n", [2, 64])
def test_block_odd_tables_bounds_and_values(pkg, gpu, n):
    model = _model(pkg, gpu, "solids", n)
    bvh = pkg.SimBVH(gpu, model)
    ren = pkg.RaycastRendererDO(gpu, model, cameraPos=(0.0, 1.6, 5.5), resolution=132)
    ren.lookAt((0.0, 0.45, 0.0))
    model.x[:, :3] += 0.01                      # bounds older than the positions
    assert _compare(pkg, gpu, model, ren) > 0
    bvh.refitBVH()
    keep = ren.dirs.clone()
    g = torch.Generator(device=gpu)
    g.manual_seed(1)
    ren.dirs.copy_(keep[torch.randperm(keep.shape[0], generator=g, device=gpu)])   # no grid
    assert _compare(pkg, gpu, model, ren) > 0
    ren.dirs.copy_(keep)
    ren.dirs[5000:9000, :3] *= 1.5              # not unit
    assert _compare(pkg, gpu, model, ren) > 0
    ren.dirs.copy_(keep)
    first = model.env_vbase[:-1]
    for k, bad in enumerate((float("nan"), float("inf"), 3e38)):
        model.x[int(first[k % n]) + 7 * k + 200, k % 3] = bad
    bvh.refitBVH()
    assert _compare(pkg, gpu, model, ren) > 0


@pytest.mark.parametrize("per_leaf", [3, 64, 10 ** 6])  # several triangles per leaf; the list overflows; the root is a leaf
def test_block_large_leaves(pkg, gpu, per_leaf):
    model = _model(pkg, gpu, "cube", 3)
    nf = model.meshes[0].num_tris
    left, first, count, level = [0], [0], [nf], [0]
    todo = [(0, 0, nf, 0)]
    while todo:                                 # halve the triangle range down to the leaf size
        k, a, n, lv = todo.pop()
        first[k], count[k], level[k], left[k] = a, n, lv, -1
        if n > per_leaf:
            left[k], count[k] = len(left), 0
            for b, m in ((a, n // 2), (a + n // 2, n - n // 2)):
                todo.append((len(left), b, m, lv + 1))
                left.append(-1), first.append(0), count.append(0), level.append(0)
    arr = lambda v: np.asarray(v, np.int32)
    model.set_bvh(0, {"left": arr(left), "first": arr(first), "count": arr(count), "level": arr(level),
                      "tri_map": np.arange(nf, dtype=np.int32), "num_nodes": len(left), "max_level": max(level)})
    pkg.SimBVH(gpu, model)
    for n_res in (20, 132):
        ren = pkg.RaycastRendererDO(gpu, model, cameraPos=(2.2, 1.8, 2.6), resolution=n_res)
        ren.lookAt((0.5, 0.45, 0.5))
        assert _compare(pkg, gpu, model, ren) > 0
