"""What tuning leaves behind: the model's partition as it was unless a
partitioned frame is the choice."""
import pytest
import torch

pytestmark = pytest.mark.gpu
KW = dict(simSubsteps=8, distance="xpbd", volume="xpbd")


def _model(pkg, gpu, tets, n):
    return pkg.SimModelDO([pkg.scenes.solid("ellipsoid", tets, seed=17)], [0] * n, device=gpu, **KW)


@pytest.mark.parametrize("own", [None, dict(tets_per_part=700, parts=None)])
def test_partition_is_as_before_when_no_parts_win(pkg, gpu, own, monkeypatch):
    A = pkg.autotune
    a, b = (_model(pkg, gpu, 9000, 6) for _ in range(2))
    if own:
        b.enable_parts(**own)
    had_default = b._default_store is not None
    # timings of a device on which one workgroup per env wins
    real = A.Autotuner._time
    monkeypatch.setattr(A.Autotuner, "_time", staticmethod(
        lambda model, cfg, frames, stream: real(model, cfg, frames, stream) + (1e3 if cfg["parts"] else 0.0)
        + (1e3 if cfg["shared"] else 0.0)))
    cfg = A.Autotuner().tune(b, frames=1)
    assert not cfg["parts"] and not cfg["shared"]
    assert b.parts_cfg == (own or {}) and (getattr(b, "_parts", None) is not None) == bool(own)
    integ = pkg.SimIntegratorDO(gpu)
    integ.stepModel(b, refit=True)              # an integrator that is not tuned
    assert (b._default_store is not None) == had_default
    pkg.lib.ffsrl_frame(a.batch, a.params, None, 1024, 1, a.stream())
    if own:
        pkg.SimIntegratorDO(gpu, parts=True).stepModel(b, refit=True)
        pkg.lib.ffsrl_frame(a.batch, a.params, None, 1024, 1, a.stream())
    torch.cuda.synchronize()
    assert torch.equal(a.x, b.x) and torch.equal(a.v, b.v)


def test_disable_parts(pkg, gpu):
    a, b = (_model(pkg, gpu, 20000, 5) for _ in range(2))
    assert b._default_store is not None
    base = torch.cuda.memory_allocated(gpu)
    integ = pkg.SimIntegratorDO(gpu)
    for k in range(3):
        b.enable_parts(tets_per_part=3000)
        assert b.default_parts() is None
        pkg.SimIntegratorDO(gpu, parts=True).stepModel(b)
        b.disable_parts()
        assert b.default_parts() is not None and b.parts_cfg == {}
        integ.stepModel(b)
        for _ in range(2):
            pkg.lib.ffsrl_frame(a.batch, a.params, None, 1024, 0, a.stream())
    torch.cuda.synchronize()
    assert torch.equal(a.x, b.x) and torch.cuda.memory_allocated(gpu) <= base + (1 << 20)


def test_choice_is_no_slower_than_no_choice(pkg, gpu, tmp_path, monkeypatch):
    """The default frame's own partition is timed, may be chosen and is then what
    the tuned integrator runs; a cache written for other kernels is not used."""
    A = pkg.autotune
    a, b = (_model(pkg, gpu, 20000, 5) for _ in range(2))
    cache = str(tmp_path / "tune.json")
    old = A.Autotuner(cache)
    old.cache[A.key_of(b).replace(f"k{A.KERNELS}", f"k{A.KERNELS - 1}")] = {
        "best": {"block": 256, "dispatch": "table", "chunk": 64, "shared": False, "parts": 0}}
    old.save()
    real = A.Autotuner._time
    monkeypatch.setattr(A.Autotuner, "_time", staticmethod(
        lambda model, cfg, frames, stream: real(model, cfg, frames, stream) + (1e3 if cfg["parts"] != "default" else 0.0)))
    integ = pkg.SimIntegratorDO(gpu)
    cfg = integ.autotune(b, cache_path=cache, frames=1)
    assert cfg["parts"] == "default" and cfg["block"] == 1024 and cfg["dispatch"] == "lpt" and not cfg["shared"]
    assert b.parts_cfg == {} and not integ.parts and not integ.tuned
    calls = []
    run = pkg.lib.ffsrl_frame_parts
    monkeypatch.setattr(type(pkg.lib), "ffsrl_frame_parts", lambda self, *x: calls.append(x[2]) or run(*x), raising=False)
    integ.stepModel(b, refit=True)
    monkeypatch.undo()
    assert len(calls) == 1
    again = pkg.SimIntegratorDO(gpu)
    assert again.autotune(b, cache_path=cache) == cfg
    again.stepModel(b, refit=True)
    for _ in range(2):
        pkg.lib.ffsrl_frame(a.batch, a.params, None, 1024, 1, a.stream())
    torch.cuda.synchronize()
    assert torch.equal(a.x, b.x) and torch.equal(a.bvh_lo, b.bvh_lo)


def test_trials_are_long_enough(pkg, gpu, monkeypatch):
    """A trial of short frames runs many of them, measured after as many that are not."""
    A = pkg.autotune
    m = _model(pkg, gpu, 900, 2)
    run, calls = pkg.lib.ffsrl_frame, []
    monkeypatch.setattr(type(pkg.lib), "ffsrl_frame", lambda self, *x: calls.append(1) or run(*x), raising=False)
    ms = A.Autotuner._time(m, dict(A.DEFAULT), 2, torch.cuda.current_stream(gpu))
    assert 0 < ms < 1.0 and (len(calls) - 2) / 2 >= min(200, A.TRIAL_MS / 1.0)
