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
