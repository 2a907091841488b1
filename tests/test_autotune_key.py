"""The autotuner's cache entries name the flux kernel that they were timed on."""
from types import SimpleNamespace

import pytest

torch = pytest.importorskip("torch")
wmx = pytest.importorskip("wmles_jax_amd")


def solver(form, n=(8, 16, 17)):
    return SimpleNamespace(precision="fp32", scheme=wmx.KEP(2), blocks=[SimpleNamespace(n=n)], kernel_form=lambda: form)


def test_entries_of_other_kernels_do_not_apply(monkeypatch):
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda *a: "card")
    key = wmx.autotune._key
    forms = ("split", "fused", "box", "curvilinear")
    assert len({key(solver(f)) for f in forms}) == len(forms)
    assert key(solver("box")) == key(solver("box")) != key(solver("box", (8, 16, 18)))
    former = f"card|fp32|KEP|{[(8, 16, 17)]}"            # entries written before kernels were named
    assert former not in {key(solver(f)) for f in forms}
    monkeypatch.setattr(wmx.autotune, "REVISION", wmx.autotune.REVISION + 1)
    newer = key(solver("box"))
    monkeypatch.undo()
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda *a: "card")
    assert newer != key(solver("box"))


def test_candidates_reach_the_lengths_that_the_plans_choose():
    assert {1, 2, 4, 6} <= {ci for ci, _ in wmx.autotune.CANDIDATES}
