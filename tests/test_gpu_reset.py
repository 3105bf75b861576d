"""resetFixedModel in one launch (ffsrl_reset_envs) against the same reset made
environment by environment with tensor operations: every state array bit for
bit, for meshes below and above one block of 256 vertices, lists of one, of
more than one launch's 500 environments, out of order and with repeats, with
and without the instrument hierarchy."""
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
FIXTURE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "liver_retraction.npz")


def _scramble(model, seed):
    g = torch.Generator(device="cpu").manual_seed(seed)
    for name in ("x", "p", "v", "drag", "laparoscopeTip", "laparoscopeBase", "laparoscopeXForm"):
        t = getattr(model, name, None)
        if t is not None:
            t.copy_(torch.rand(t.shape, generator=g).to(t.device))
    for name in ("laparoscopeDragCutHeat", "laparoscopeDragCutHeatUpdate"):
        t = getattr(model, name, None)
        if t is not None:
            t.fill_(1)


def _state(model):
    names = ("x", "p", "v", "drag", "laparoscopeTip", "laparoscopeBase", "laparoscopeXForm", "laparoscopeDragCutHeat",
             "laparoscopeDragCutHeatUpdate")
    return {k: getattr(model, k).cpu().numpy().copy() for k in names if getattr(model, k, None) is not None}


@pytest.mark.parametrize("instrument", [False, True])
@pytest.mark.parametrize("ids", [[0], [5, 2, 2, 7], list(range(8)), [i % 8 for i in range(1003)], []])
def test_one_launch_equals_the_reset_env_by_env(pkg, gpu, instrument, ids):
    if instrument:
        m = pkg.SimModelDO.from_usd(FIXTURE, 8, device=gpu, distance="pbd", volume="pbd")
    else:
        meshes = [pkg.scenes.cube_grid(c) for c in (2, 4, 7)]  # 8, 64 and 343 vertices
        tips = np.random.default_rng(2).random((8, 4, 3)).astype(np.float32)
        m = pkg.SimModelDO(meshes, [i % 3 for i in range(8)], device=gpu, tips=tips, distance="pbd", volume="pbd")
    m.initialVertex[:, 3] = torch.rand(m.numVertices, device=gpu)
    _scramble(m, 1)
    assert m._reset_in_one(ids)
    m.resetFixedModel(ids)
    one = _state(m)
    _scramble(m, 1)
    m._reset_in_one = lambda ids: False
    m.resetFixedModel(ids)
    for k, v in _state(m).items():
        assert np.array_equal(one[k], v), k


def test_other_lists_and_arrays_take_the_loop(pkg, gpu):
    m = pkg.SimModelDO([pkg.scenes.cube_grid(3)], [0] * 3, device=gpu, distance="pbd", volume="pbd")
    assert not m._reset_in_one([-1]) and not m._reset_in_one([3])
    with pytest.raises(IndexError):
        m.resetFixedModel([3])
    m.initialVertex = m.initialVertex.double()
    assert not m._reset_in_one([0])
    m.x.fill_(2.0)
    m.resetFixedModel([1])
    s = m.env_slice(1)
    assert torch.equal(m.x[s], m.initialVertex[s].float()) and bool((m.x[:s.start] == 2.0).all())
