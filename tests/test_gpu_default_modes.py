"""The default frame after the model's parameters have been set to other
constraints than it was built with: its partition follows them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("built,change", [
    (dict(distance=None, volume="pbd"), dict(dist_mode=1, dist_k=1.0)),
    (dict(distance="pbd", volume=None), dict(vol_mode=1, vol_k=1.0)),
    (dict(distance="pbd", volume="pbd"), dict(dist_mode=0)),
    (dict(distance="pbd", volume=None), dict(vol_mode=1, vol_k=1.0, dist_mode=0, iterations=2)),
    (dict(distance="pbd", volume="pbd"), dict(nh_on=1)),
])
def test_default_frame_follows_the_parameters(pkg, gpu, built, change):
    mesh = pkg.scenes.solid("ellipsoid", 14000, seed=91)
    a, b = (pkg.SimModelDO([mesh], [0, 0], device=gpu, simSubsteps=6, **built) for _ in range(2))
    assert b.default_parts() is not None
    for m in (a, b):
        g = torch.Generator(device=gpu)
        g.manual_seed(2)
        m.v[:, :3] = 0.2 * torch.randn((m.numVertices, 3), generator=g, device=gpu)
    integ = pkg.SimIntegratorDO(gpu)
    for f in range(3):
        if f:
            for m in (a, b):
                for k, v in change.items():
                    setattr(m.params, k, v)
        pkg.lib.ffsrl_frame(a.batch, a.params, a.dispatch_order().data_ptr(), 1024, 1, a.stream())
        integ.stepModel(b, refit=True)
        torch.cuda.synchronize()
        assert all(torch.equal(getattr(a, k), getattr(b, k)) for k in ("x", "v", "p", "bvh_lo", "bvh_hi")), f
    assert int(b.frame_status().abs().sum()) == 0
