"""The partitioned frame's assembly (ff-srl_amd/csrc/parts_wait.hpp) run by
host threads: either every part of an env goes on or every part withdraws; an
env that only its parts can run is not given up because the XCD is idle."""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "ff-srl_amd"))


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    import build as B
    hipcc = B._hipcc()
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    exe = str(tmp_path_factory.mktemp("wait") / "parts_wait_harness")
    r = subprocess.run([hipcc, *[f for f in B.HIPCC_FLAGS if f != "-fPIC"], "-pthread",
                        os.path.join(ROOT, "tests", "parts_wait_harness.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return exe


@pytest.mark.parametrize("parts", [2, 5])
@pytest.mark.parametrize("scenario,rounds", [("all", 200), ("absent", 200), ("race", 1000), ("busy", 20), ("large", 20),
                                             ("limit", 200)])
def test_parts_agree(harness, scenario, rounds, parts):
    r = subprocess.run([harness, scenario, str(parts), str(rounds)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    _, went, _, left = r.stdout.split()
    assert int(went) + int(left) == rounds
    if scenario == "race":   # both ends were reached
        assert int(went) > 0 and int(left) > 0


@pytest.mark.gpu
def test_withdrawn_env_without_another_form_is_reported(pkg, gpu):
    """An env above the one-workgroup frame's vertex limit whose parts withdrew
    (the flag set from the host): reported as incomplete, its state as before,
    sums and counters left at zero; the next frame runs it."""
    import torch
    m = pkg.SimModelDO([pkg.scenes.cube_grid(23)], [0], device=gpu, distance="pbd", volume="pbd", simSubsteps=3)
    assert m.max_nv > pkg.lib.ffsrl_frame_max_vertices()
    m.enable_parts()
    x = m.x.clone()
    m.p_ctr[3] = -2**31
    integ = pkg.SimIntegratorDO(gpu, parts=True)
    integ.stepModel(m)
    torch.cuda.synchronize()
    assert int(m.frame_status()[0]) == pkg._lib.STATUS_INCOMPLETE and torch.equal(m.x, x)
    assert int(m.p_ctr[:4 + 32].abs().sum()) == 0 and int(m.p_sums.abs().sum()) == 0
    m.clear_status()
    integ.stepModel(m)
    torch.cuda.synchronize()
    assert int(m.frame_status()[0]) == 0 and not torch.equal(m.x, x) and np.isfinite(m.x.cpu().numpy()).all()
