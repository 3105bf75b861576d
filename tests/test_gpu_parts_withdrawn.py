"""Envs whose parts withdrew from a partitioned frame (they could not all run
at once) are run by one workgroup in the launch behind it.  The flag is set
from the host before the launch, so every part of those envs finds it and goes
on; state, carried multipliers, contact counts, bounds and status equal the
one-workgroup frame bit for bit, and the counters are left at zero."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
BASE = dict(simSubsteps=5, simFrameRate=60, environmentGravity=(0.0, -9.81, 0.0), environmentVelocityDampening=0.1,
            distance="xpbd", volume="xpbd", distanceCompliance=1e-6, volumeComplianceXPBD=0.0, globalKsDrag=1.0)


@pytest.mark.parametrize("collision", [False, True])
@pytest.mark.parametrize("iterations", [1, 2])
@pytest.mark.parametrize("withdrawn", [[1], [0, 3, 4], [0, 1, 2, 3, 4]])
def test_withdrawn_envs_equal_the_one_workgroup_frame(pkg, gpu, collision, iterations, withdrawn):
    sc = pkg.scenes
    meshes = [sc.solid("ellipsoid" if i % 2 else "box", t, seed=31 + i) for i, t in enumerate((9000, 4000, 1200, 30000, 6000))]
    tips = np.stack([np.repeat((sc.top_point(m) + np.array([0.0, 0.02, 0.0], np.float32))[None], 4, axis=0)
                     for m in meshes]).astype(np.float32)
    kw = dict(BASE, simConstraintsSteps=iterations, tips=tips)
    if collision:
        # a capsule of radius 0.12 over each env's highest vertex, pressed 0.036 deep
        low = tips + np.array([0.0, -0.056, 0.0], np.float32)
        kw.update(collision=True, globalKsContact=1.0, capsuleBases=low, tips=low + np.array([0.0, 0.62, 0.0], np.float32),
                  capsuleRadii=np.tile(np.array([0.12, 0.0, 0.0, 0.0], np.float32), (len(meshes), 1)))
    a, b = (pkg.SimModelDO(meshes, list(range(5)), device=gpu, **kw) for _ in range(2))
    b.enable_parts(tets_per_part=2000)
    order = a.dispatch_order().data_ptr()
    for frame in range(3):
        if frame:  # the first frame without: the words must also be left clean by a frame like that
            for e in withdrawn:
                if b._parts_host[e, 1] > 1:
                    b.p_ctr[4 * e + 3] = -2**31
        pkg.lib.ffsrl_frame(a.batch, a.params, order, 1024, 1, a.stream())
        pkg.lib.ffsrl_frame_parts(b.batch, b.params, b.parts, order, 5, 1, b.stream())
        torch.cuda.synchronize()
        for k in ("x", "v", "p", "bvh_lo", "bvh_hi", "status", "laparoscopeInCollision", "lam_t", "lam_e"):
            ta, tb = getattr(a, k), getattr(b, k)
            assert (ta is None and tb is None) or torch.equal(ta, tb), (frame, k)
        assert int(b.frame_status().abs().sum()) == 0
        assert int(b.p_ctr[:4 * 5 + 32].abs().sum()) == 0 and int(b.p_sums.abs().sum()) == 0
    if collision:
        assert int(a.laparoscopeInCollision.sum()) > 0
