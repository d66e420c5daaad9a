"""Saved winners of the autotuner: those timed on another launch of the batched
trace are not taken for the present one."""
import json
from types import SimpleNamespace

from turbulence_tracing_amd import autotune
from turbulence_tracing_amd.ensemble import Ensemble, Member


def test_winners_of_the_queue_launch_are_timed_again(tmp_path, monkeypatch):
    monkeypatch.setattr(autotune, "device_key", lambda device=None: "gfx950:256cu")
    members = [Member(n=128, beta=-3.4, aniso=1.0, rms=0.1, ne0=1e24, n_rays=1000, seed=0)]
    ens = SimpleNamespace(members=members, h=0.5)
    old = {"members": [(128, 1000)], "h": 0.5}  # the signature winners were saved under before
    path = tmp_path / "autotune.json"
    best = {"block": 256, "blocks_per_cu": 2, "variant": 0, "chunk": 256, "brick_shift": 0}
    path.write_text(json.dumps({autotune.Autotuner.key("ensemble_trace", old): {"best": best, "ms": 1.0, "all": []}}))
    tuner = autotune.Autotuner(str(path))
    assert tuner.report("ensemble_trace", old)["best"] == best
    assert tuner.report("ensemble_trace", Ensemble.signature(ens)) is None
    # one and the same for the same ensemble, others for others
    assert Ensemble.signature(ens) == Ensemble.signature(SimpleNamespace(members=list(members), h=0.5))
    assert Ensemble.signature(ens) != Ensemble.signature(SimpleNamespace(members=members, h=0.25))
