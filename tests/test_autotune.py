"""The launch sweep of amr.autotune on the CPU, with the launches and their timing replaced."""
import itertools
import types

import pytest

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("scheme,shapes", [("MHM_RP", {"4", "8"}), ("MHM", {"4"})])
def test_every_launch_is_timed_once_a_round(monkeypatch, scheme, shapes):
    """The accepted workgroup shapes run the same kernel: their configurations share one time, so that the choice between
    them is no noise, and the sweep does not time a launch twice."""
    from gamer_amd import amr, hydro
    calls, clock = [], itertools.count(1)
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda i: "cpu")
    monkeypatch.setattr(hydro, "solve_batch", lambda u, pg, **kw: calls.append(
        (kw.get("queue_counter") is not None, kw.get("groups_per_cu"), kw.get("pgs_per_ticket"), kw["waves_per_group"])))

    def time_launch(torch_, fn, reps):
        n = len(calls)
        fn()
        timed.append(calls[n][:3])
        return 1.0 / next(clock)
    timed = []
    monkeypatch.setattr(amr, "time_launch", time_launch)
    batch = types.SimpleNamespace(u=torch.zeros((2, 5, 1, 1, 1)), pg_dt_dh=torch.zeros((2, 2)))
    res = amr.autotune(torch, batch, groups=(1, 2), tickets=(1, 2), rounds=3, scheme=scheme)
    assert len(timed) == 15 and all(timed.count(t) == 3 for t in timed)
    assert {c[3] for c in calls} == {int(s) for s in shapes}                   # every shape was accepted by a launch
    names = {f"{m}:{s}" for m in ["grid"] + [f"persistent:{g}:{k}" for g in (1, 2) for k in (1, 2)] for s in shapes}
    assert set(res["trials_ms"]) == names and res["best"] in names
    for m in {n.rpartition(":")[0] for n in names}:
        assert len({res["trials_ms"][f"{m}:{s}"] for s in shapes}) == 1
