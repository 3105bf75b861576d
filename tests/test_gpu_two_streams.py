"""Two models stepped by the default integrator on two streams at once: their
parts share the CUs (and may withdraw from an env that they cannot run at
once); each model's state equals its one-workgroup frames bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tets,envs", [((9000, 4000), 40), ((30000, 20000), 24)])
def test_two_models_on_two_streams(pkg, gpu, tets, envs):
    kw = dict(simSubsteps=4, simFrameRate=60, distance="xpbd", volume="xpbd", distanceCompliance=1e-6,
              volumeComplianceXPBD=0.0)
    meshes = [pkg.scenes.solid("ellipsoid", t, seed=71 + i) for i, t in enumerate(tets)]
    ref, got = ([pkg.SimModelDO([m], [0] * (envs + 7 * i), device=gpu, **kw) for i, m in enumerate(meshes)]
                for _ in range(2))
    assert all(m.default_parts() is not None and m.default_parts().max_local > 0 for m in got)
    streams = [torch.cuda.Stream(gpu) for _ in got]
    orders = [m.dispatch_order() for m in ref + got]
    torch.cuda.synchronize()
    integ = pkg.SimIntegratorDO(gpu)
    for _ in range(15):
        for m, s in zip(got, streams):
            with torch.cuda.stream(s):
                integ.stepModel(m, refit=True)
    torch.cuda.synchronize()
    for m, o in zip(ref, orders):
        for _ in range(15):
            pkg.lib.ffsrl_frame(m.batch, m.params, o.data_ptr(), 1024, 1, m.stream())
    torch.cuda.synchronize()
    for a, b in zip(ref, got):
        assert int(b.frame_status().abs().sum()) == 0
        assert all(torch.equal(getattr(a, k), getattr(b, k)) for k in ("x", "v", "p", "bvh_lo", "bvh_hi"))


@pytest.mark.parametrize("mode", ["nh", "xpbd", "collision"])
@pytest.mark.parametrize("listed", [False, True])
def test_every_env_in_one_part(pkg, gpu, mode, listed):
    """Envs of one part each, listed or not, at the largest size and the smallest."""
    sc = pkg.scenes
    meshes = [sc.solid("ellipsoid", 20000, seed=81), sc.solid("box", 40, seed=82), sc.solid("box", 2000, seed=83)]
    assert pkg.lib.ffsrl_parts_max_solo() - 64 < meshes[0].num_vertices <= pkg.lib.ffsrl_parts_max_solo()
    kw = dict(simSubsteps=3, simConstraintsSteps=2, distance="xpbd", volume="xpbd", neoHookean=mode == "nh")
    if mode == "collision":
        low = torch.stack([torch.from_numpy(sc.top_point(m)) for m in meshes for _ in range(4)]).reshape(3, 4, 3).float()
        low[..., 1] -= 0.036
        low = low.repeat(3, 1, 1)
        kw.update(collision=True, globalKsContact=1.0, capsuleBases=low.numpy(), tips=(low + torch.tensor([0.0, 0.62, 0.0])).numpy(),
                  capsuleRadii=torch.tensor([0.12, 0, 0, 0]).repeat(9, 1).numpy())
    a, b = (pkg.SimModelDO(meshes, [0, 1, 2] * 3, device=gpu, **kw) for _ in range(2))
    b.enable_parts(tets_per_part=1 << 30)
    assert b.parts.max_local == 0
    order = torch.tensor([7, 0, 4, 8, 3], dtype=torch.int32, device=gpu) if listed else None
    for _ in range(3):
        if listed:
            pkg.lib.ffsrl_frame_envs(a.batch, a.params, order.data_ptr(), 5, 1024, 1, a.stream())
            pkg.lib.ffsrl_frame_parts(b.batch, b.params, b.parts, order.data_ptr(), 5, 1, b.stream())
        else:
            pkg.lib.ffsrl_frame(a.batch, a.params, None, 1024, 1, a.stream())
            pkg.lib.ffsrl_frame_parts(b.batch, b.params, b.parts, None, 9, 1, b.stream())
    torch.cuda.synchronize()
    for k in ("x", "v", "p", "bvh_lo", "bvh_hi", "status", "laparoscopeInCollision", "lam_t", "lam_e"):
        s, t = getattr(a, k), getattr(b, k)
        assert (s is None and t is None) or torch.equal(s, t), k
    if mode == "collision":
        assert int(a.laparoscopeInCollision.sum()) > 0


@pytest.mark.parametrize("large", [False, True])
def test_frame_beside_a_launch_that_holds_the_cus(pkg, gpu, large):
    """Another stream's frame holds all but a few CUs for about 20 ms: parts that
    cannot come together beside it withdraw and their envs are run by one
    workgroup each; an env that only its parts can run waits for the CUs."""
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    hold = pkg.SimModelDO([pkg.scenes.solid("ellipsoid", 20000, seed=5)], [0] * (cus - 8), device=gpu, simSubsteps=400,
                          distance="pbd", volume="pbd")
    kw = dict(simSubsteps=6, distance="pbd", volume="pbd")
    mesh = pkg.scenes.cube_grid(23) if large else pkg.scenes.solid("ellipsoid", 20000, seed=6)
    n = 2 if large else 16
    ref, got = (pkg.SimModelDO([mesh], [0] * n, device=gpu, default_partition=False, **kw) for _ in range(2))
    for m in (ref, got):
        m.enable_parts(tets_per_part=1 << 30 if large else 1280)
        assert int(m._parts_host[:, 1].max()) > 2 and (m.max_nv > pkg.lib.ffsrl_frame_max_vertices()) == large
    integ = pkg.SimIntegratorDO(gpu, parts=True)
    orders = [m.dispatch_order() for m in (hold, ref, got)]
    a, b = torch.cuda.Stream(gpu), torch.cuda.Stream(gpu)
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        pkg.lib.ffsrl_frame(hold.batch, hold.params, orders[0].data_ptr(), 1024, 0, hold.stream())
    with torch.cuda.stream(b):
        for _ in range(2):
            integ.stepModel(got, refit=True)
    torch.cuda.synchronize()
    for _ in range(2):                      # the device to itself
        integ.stepModel(ref, refit=True)
    torch.cuda.synchronize()
    assert int(got.frame_status().abs().sum()) == 0 and int(got.p_ctr[:4 * n + 32].abs().sum()) == 0
    assert int(got.p_sums.abs().sum()) == 0
    assert all(torch.equal(getattr(ref, k), getattr(got, k)) for k in ("x", "v", "p", "bvh_lo", "bvh_hi"))
