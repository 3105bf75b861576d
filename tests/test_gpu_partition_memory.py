"""Device memory of the partitions: no sums where every env is in one part, one
partition at a time, and none for a server that does not use the default's."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
KW = dict(simSubsteps=2, distance="xpbd", volume="xpbd", neoHookean=True)


def test_envs_in_one_part_hold_no_sums(pkg, gpu):
    n = torch.cuda.get_device_properties(gpu).multi_processor_count
    mesh = pkg.scenes.solid("box", 900, seed=4)
    a, m = (pkg.SimModelDO([mesh], [0] * n, device=gpu, **KW) for _ in range(2))
    st = m._default_store
    assert st is not None and st.pt.max_local == 0 and st.p_sums.numel() == 6
    base = torch.cuda.memory_allocated(gpu)
    m.enable_parts(tets_per_part=1 << 30)
    assert m._default_store is None and m.p_sums.numel() == 6
    m.enable_parts(tets_per_part=300)            # sums are needed now
    assert m.p_sums.shape == (3, m.numVertices, 2) and m.parts.stride == m.numVertices
    integ = pkg.SimIntegratorDO(gpu, parts=True)
    for per in (300, 1 << 30, 300):
        m.enable_parts(tets_per_part=per)
        pkg.lib.ffsrl_frame(a.batch, a.params, None, 1024, 0, a.stream())
        integ.stepModel(m)
        torch.cuda.synchronize()
        assert torch.equal(a.x, m.x) and int(m.frame_status().abs().sum()) == 0
    assert base > 0


def test_enable_parts_frees_the_default_partition_first(pkg, gpu):
    mesh = pkg.scenes.solid("ellipsoid", 20000, seed=4)
    m = pkg.SimModelDO([mesh], [0] * 40, device=gpu, simSubsteps=10)
    assert m.default_parts().max_local > 0
    torch.cuda.reset_peak_memory_stats(gpu)
    before = torch.cuda.memory_allocated(gpu)
    m.enable_parts(tets_per_part=5120)
    # the same sums and about the same tables in their place: well below two sets
    assert torch.cuda.max_memory_allocated(gpu) - before < 24 * m.numVertices


def test_server_builds_no_default_partition(pkg, gpu):
    mesh = pkg.scenes.solid("ellipsoid", 6000, seed=4)
    tips = np.zeros((1, 4, 3), np.float32)
    s = pkg.serve.SceneServer([mesh], [8], 1e9, dict(KW, neoHookean=False, simSubsteps=10), tips, device=gpu)
    assert s.model._default_store is None
    t = pkg.serve.SceneServer([mesh], [8], 1e9, dict(KW, neoHookean=False, simSubsteps=10, default_partition=True), tips,
                              device=gpu)
    assert t.model._default_store is not None
    a, b = s.model, t.model                       # the first frame that uses it builds it
    integ = pkg.SimIntegratorDO(gpu)
    integ.stepModel(a)
    integ.stepModel(b)
    torch.cuda.synchronize()
    assert a._default_store is not None and torch.equal(a.x, b.x)
