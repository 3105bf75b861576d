"""The default frame's own partition: the rule that chooses it (host), and on
the GPU the default integrator against ffsrl_frame called directly: state,
carried multipliers, contact counts, bounds and status bit for bit."""
import numpy as np
import pytest
import torch

STATE = ("x", "v", "p", "bvh_lo", "bvh_hi", "status", "laparoscopeInCollision", "lam_t", "lam_e")
BASE = dict(simSubsteps=4, simFrameRate=60, environmentGravity=(0.0, -9.81, 0.0), environmentVelocityDampening=0.1,
            distanceCompliance=1e-6, volumeComplianceXPBD=0.0, globalKsDrag=1.0, globalVolumeCompliance=1.0 / 5e4,
            globalDeviatoricCompliance=1.0 / 1e4)
MODES = {
    "pbd": dict(distance="pbd", volume="pbd"),
    "edges": dict(distance="pbd", volume=None),
    "tets": dict(distance=None, volume="pbd"),
    "nh": dict(distance="xpbd", volume="xpbd", neoHookean=True),
    "xpbd-i2": dict(distance="xpbd", volume="xpbd", simConstraintsSteps=2),
    "nh-i3": dict(distance="xpbd", volume="xpbd", neoHookean=True, simConstraintsSteps=3, simSubsteps=2),
    "xpbd-legacy": dict(distance="xpbd", volume="xpbd", lambdaLegacy=True),
}


def _rule(pkg, items, env_mesh, cus=256, nxcd=8, collision=False):
    import importlib
    f = importlib.import_module("ff-srl_amd.model").default_tets_per_part
    return f(items, [max(8, t // 4) for t in items], env_mesh, cus, nxcd, collision)


@pytest.mark.parametrize("items,env_mesh,kw,parts", [
    ([], [], {}, False),                                       # no env
    ([0], [0], {}, False),                                     # nothing to cut
    ([1], [0], {}, False),
    ([1280], [0], {}, False), ([1281], [0], {}, False),        # a cut would not pay its exchange
    ([4000], [0], {}, True), ([20000], [0], {}, True),
    ([20000], [0] * 256, {}, False),                           # every CU has its env
    ([20000], [0] * 300, {}, True),                            # the last 44 run alone
    ([20000], [0] * 512, {}, False), ([20000], [0] * 5000, {}, False),
    ([40000, 1000], [0] + [1] * 255, {}, True),
    ([40000], [0] * 9, dict(cus=32, nxcd=1), True),            # a device partition
    ([40000], [0] * 4, dict(cus=4, nxcd=4), False),            # one CU per XCD: no part has company
    ([40000], [0], dict(nxcd=0), False),                       # XCDs unknown
    ([20000, 2000], [0, 1] * 20, dict(collision=True), True),
])
def test_rule(pkg, items, env_mesh, kw, parts):
    assert (_rule(pkg, items, env_mesh, **kw) is not None) == parts


def _models(pkg, gpu, mode, collision, n=2, seed=41):
    sc = pkg.scenes
    meshes = [sc.solid("ellipsoid" if i % 2 else "box", t, seed=seed + i) for i, t in enumerate((16000, 900, 5000))]
    tips = np.stack([np.repeat((sc.top_point(m) + np.array([0.0, 0.02, 0.0], np.float32))[None], 4, axis=0)
                     for m in meshes]).astype(np.float32)
    kw = dict(BASE, **MODES[mode])
    if collision:
        low = tips + np.array([0.0, -0.056, 0.0], np.float32)
        kw.update(collision=True, globalKsContact=1.0, capsuleBases=low,
                  capsuleRadii=np.tile(np.array([0.12, 0.0, 0.0, 0.0], np.float32), (3, 1)))
        tips = low + np.array([0.0, 0.62, 0.0], np.float32)
    out = []
    for _ in range(n):
        m = pkg.SimModelDO(meshes, [0, 1, 2], device=gpu, tips=tips, **kw)
        m.v[:, :3] = torch.from_numpy(np.random.default_rng(3).uniform(-0.05, 0.05, (m.numVertices, 3))).to(m.v)
        if not collision:
            m.set_grasp(0, sc.nearest_surface_vertices(meshes[0], tips[0, 2], 8))
        out.append(m)
    return out


def _frames(pkg, gpu, a, b, k=2, refit=True):
    integ = pkg.SimIntegratorDO(gpu)
    for _ in range(k):
        pkg.lib.ffsrl_frame(a.batch, a.params, a.dispatch_order().data_ptr(), 1024, int(refit), a.stream())
        integ.stepModel(b, refit=refit)
    torch.cuda.synchronize()
    for name in STATE:
        ta, tb = getattr(a, name), getattr(b, name)
        assert (ta is None and tb is None) or torch.equal(ta, tb), name


@pytest.mark.gpu
@pytest.mark.parametrize("collision", [False, True])
@pytest.mark.parametrize("mode", list(MODES))
def test_default_frame_equals_one_workgroup_per_env(pkg, gpu, mode, collision):
    a, b = _models(pkg, gpu, mode, collision)
    assert b.default_parts() is not None and b.default_parts().max_local > 0
    _frames(pkg, gpu, a, b)
    assert int(b._default_store.p_ctr[:4 * 3 + 32].abs().sum()) == 0 and int(b._default_store.p_sums.abs().sum()) == 0
    for m in (a, b):  # the partition follows the constraint order
        m.set_constraint_order("local", 64)
    _frames(pkg, gpu, a, b, refit=False)
    if collision:
        assert int(a.laparoscopeInCollision.sum()) > 0


@pytest.mark.gpu
def test_what_keeps_one_workgroup_per_env(pkg, gpu):
    """Capture, a partition of the model's own, other launch shapes; a mesh
    above the one-workgroup limit stays refused."""
    a, b = _models(pkg, gpu, "pbd", False)
    s = torch.cuda.Stream(gpu)
    g = torch.cuda.CUDAGraph()
    b.dispatch_order()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        assert b.default_parts() is None
        pkg.SimIntegratorDO(gpu).stepModel(b, refit=True)
    for _ in range(3):
        pkg.lib.ffsrl_frame(a.batch, a.params, a.dispatch_order().data_ptr(), 1024, 1, a.stream())
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(getattr(a, k), getattr(b, k)) for k in ("x", "v", "p", "bvh_lo", "bvh_hi"))
    b.set_constraint_order("local", 64)  # in place: the captured frame stays valid
    a.set_constraint_order("local", 64)
    pkg.lib.ffsrl_frame(a.batch, a.params, a.dispatch_order().data_ptr(), 1024, 1, a.stream())
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(a.x, b.x)
    for integ in (pkg.SimIntegratorDO(gpu, block=512), pkg.SimIntegratorDO(gpu, dispatch_sorted=False)):
        integ.stepModel(b)
    tuned = pkg.SimIntegratorDO(gpu)
    tuned.configure({"block": 1024, "dispatch": "lpt"})
    tuned.stepModel(b)
    assert b._default_store is not None
    b.enable_parts()
    assert b.default_parts() is None and b._default_store is None
    big = pkg.SimModelDO([pkg.scenes.cube_grid(23)], [0], device=gpu, distance="pbd", volume="pbd")
    assert big.max_nv > pkg.lib.ffsrl_frame_max_vertices() and big.default_parts() is None
    with pytest.raises(pkg.FFSRLError, match="ffsrl_frame failed"):
        pkg.SimIntegratorDO(gpu).stepModel(big)


@pytest.mark.gpu
@pytest.mark.parametrize("collision,iterations,parts", [(False, 1, True), (False, 2, True), (True, 1, True), (True, 2, False)])
def test_full_chip_of_whole_envs(pkg, gpu, collision, iterations, parts):
    """At least as many Neo-Hookean envs as CUs, each within one part's LDS."""
    n = torch.cuda.get_device_properties(gpu).multi_processor_count
    n += -n % 8
    mesh = pkg.scenes.solid("box", 600, seed=3)
    tip = np.repeat((pkg.scenes.top_point(mesh) + np.array([0.0, 0.02, 0.0], np.float32))[None], 4, axis=0)
    kw = dict(BASE, distance="xpbd", volume="xpbd", neoHookean=True, simConstraintsSteps=iterations,
              tips=np.tile(tip[None], (n, 1, 1)).astype(np.float32))
    if collision:
        kw.update(collision=True, globalKsContact=1.0, capsuleBases=kw["tips"] + np.array([0.0, 0.5, 0.0], np.float32),
                  capsuleRadii=np.full((n, 4), 0.03, np.float32))
    a, b = (pkg.SimModelDO([mesh], [0] * n, device=gpu, **kw) for _ in range(2))
    pt = b.default_parts()
    assert (pt is not None) == parts and (pt is None or pt.max_local == 0)
    _frames(pkg, gpu, a, b)


@pytest.mark.parametrize("items,env_mesh,passes,parts", [
    ([4000], [0], 1, False), ([4000], [0], 2, False), ([4000], [0], 4, True),
    ([4000], [0] * 100, 2, False), ([4000], [0] * 100, 4, False), ([4000], [0] * 100, 8, True),
    ([6000], [0] * 30, 1, False), ([6000], [0] * 100, 2, False), ([6000], [0] * 100, 4, True),
    ([9000], [0] * 100, 1, False), ([9000], [0] * 100, 2, True), ([20000], [0] * 100, 1, False),
    ([20000], [0], 1, True), ([20000], [0] * 30, 1, True), ([30000, 12000, 5000, 2000], [0, 1, 2, 3] * 125, 1, False),
])
def test_rule_few_passes(pkg, items, env_mesh, passes, parts):
    """Parts start and end once a frame: a frame of few passes must win that back."""
    import importlib
    f = importlib.import_module("ff-srl_amd.model").default_tets_per_part
    assert (f(items, [t // 4 for t in items], env_mesh, 256, 8, False, passes) is not None) == parts
