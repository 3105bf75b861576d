"""The frame's fixed-point terms on both sides of 2^22 quanta, where the
conversion changes from one biased float add to the clamping one, up to the
2^24 quanta at which a term saturates.

One Jacobi pass over a cube stretched by 1 + s about its centre (diagonal
sqrt(3), so a quantum is 2^-26: 2^22 quanta are 1/16 and 2^24 are 1/4); the PBD
distance terms that saturate follow from the stretches and inverse masses.
The plain form sums floats.  A term's rounding is at most half a quantum and the
mean of the terms no more, 4e-9 of the diagonal; the hardware reciprocals and
square roots add a few ulp (6e-8) of terms of at most a quarter: 1e-6 of the
diagonal bounds both."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [2, 5])
@pytest.mark.parametrize("form", ["batched", "batched256", "shared", "parts"])
@pytest.mark.parametrize("s", [-0.05, 0.06, 0.0883, 0.0885, 0.1249, 0.1251, 0.2, 0.35, 0.6])
def test_terms_around_the_conversion_limits(pkg, gpu, cells, form, s):
    mesh = pkg.scenes.cube_grid(cells)
    scale = 1.0 if cells == 2 else (cells - 1.0)  # of the stretch, so that an edge's term is that of one cell
    kw = dict(simSubsteps=1, simConstraintsSteps=1, simFrameRate=60, environmentGravity=(0.0, 0.0, 0.0),
              environmentVelocityDampening=0.0, environmentGroundLevel=-100.0, distance="pbd", volume=None,
              globalKsDistance=1.0)
    out = []
    for f in (form, "plain"):
        m = pkg.SimModelDO([mesh], [0, 0], device=gpu, **kw)
        c = m.x[:, :3].mean(0)
        m.x[:, :3] = c + (m.x[:, :3] - c) * (1.0 + s * scale)
        if f == "parts":
            m.enable_parts(parts=[2])
        integ = pkg.SimIntegratorDO(gpu, block=256 if f == "batched256" else 1024, shared=f == "shared", parts=f == "parts")
        integ.stepModelPlain(m) if f == "plain" else integ.stepModel(m)
        torch.cuda.synchronize()
        out.append((m.vertex().cpu().numpy().astype(np.float64), m.frame_status().cpu().numpy()))
    (x, status), (ref, _) = out
    a, b = mesh.edges[:, 0], mesh.edges[:, 1]
    w = m.initialVertex[:mesh.num_vertices, 3].cpu().numpy().astype(np.float64)
    rest = np.linalg.norm((mesh.verts[b] - mesh.verts[a]).astype(np.float64), axis=1)
    free = w[a] + w[b] > 0.0
    share = np.maximum(w[a], w[b])[free] / (w[a] + w[b])[free]
    unit = np.abs((mesh.verts[b] - mesh.verts[a])[free]).max(axis=1) / rest[free]  # largest component of the direction
    saturated = bool((np.abs(s * scale) * rest[free] * share * unit).max() > (2**24 - 1) * 2.0**-26)
    assert bool(status.any()) == saturated, (s, status)
    if not saturated:
        assert np.abs(x - ref).max() <= 1e-6 * mesh.bbox_diagonal()
