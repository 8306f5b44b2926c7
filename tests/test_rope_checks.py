"""The RoPE wrapper's one-test acceptance of usual inputs (_plain, _plain_kv) accepts nothing that its checks one by one
refuse: over stand-in tensors with one or two properties changed at a time, on the CPU."""

import itertools

import pytest
import torch


class Stub:
    def __init__(self, shape, dtype, device="cuda:0", contiguous=True):
        self.shape, self.dtype, self.device = torch.Size(shape), dtype, torch.device(device)
        self._contiguous = contiguous

    def dim(self):
        return len(self.shape)

    def is_contiguous(self):
        return self._contiguous


BF, FP, I64, F32 = torch.bfloat16, torch.float16, torch.int64, torch.float32
USUAL = {"q": ((2, 3, 8, 64), BF), "k": ((2, 3, 2, 64), BF), "v": ((2, 3, 2, 64), BF), "position_ids": ((2, 3), I64),
         "inv_freq": ((32,), F32), "k_cache": ((9, 2, 64), BF), "v_cache": ((9, 2, 64), BF), "slot_mapping": ((2, 3), I64)}
CHANGES = [("q", (2, 3, 8, 63), BF), ("q", (2, 3, 8, 62), BF), ("q", (2, 4, 8, 64), BF), ("q", (6, 8, 64), BF),
           ("q", (2, 3, 8, 64), F32), ("q", (2, 3, 8, 64), FP), ("k", (2, 3, 2, 64), FP), ("k", (2, 3, 2, 32), BF),
           ("k", (3, 2, 2, 64), BF), ("v", (2, 3, 1, 64), BF), ("v", (2, 3, 2, 64), FP), ("position_ids", (6,), I64),
           ("position_ids", (2, 3), torch.int32), ("inv_freq", (64,), F32), ("inv_freq", (32, 1), F32),
           ("inv_freq", (32,), BF), ("k_cache", (9, 2, 32), BF), ("k_cache", (8, 2, 64), BF), ("k_cache", (9, 2, 64), FP),
           ("v_cache", (9, 128), BF), ("slot_mapping", (2, 3), torch.int32), ("slot_mapping", (3, 2), I64)]


@pytest.fixture(scope="module")
def rope(pkg):
    return pkg.candidate("rope")


def _outcome(rope, monkeypatch, tensors, inplace, plain):
    """What run() does with the tensors up to the launch: the ValueError's text, or "accepted"."""
    calls = []
    with monkeypatch.context() as m:
        if not plain:
            m.setattr(rope, "_plain", lambda *a: False)
            m.setattr(rope, "_plain_kv", lambda *a: False)
        for t in tensors.values():
            def contiguous():
                calls.append(1)
                raise StopIteration  # the first thing after the checks
            t.contiguous = contiguous
        try:
            rope.run({**tensors, "inplace": inplace})
        except ValueError as e:
            return str(e)
        except StopIteration:
            return "accepted"
    return "unexpected"


def test_plain_accepts_what_the_checks_accept(rope, monkeypatch):
    kv = list(USUAL)
    freq = ["q", "k", "position_ids", "inv_freq"]
    seen = set()
    changes = [()] + [(c,) for c in CHANGES] + list(itertools.combinations(CHANGES, 2))
    for change in changes:
        for names, inplace in ((kv, False), (kv, True), (freq, False), (freq, True)):
            spec = dict(USUAL)
            for name, shape, dtype in change:
                spec[name] = (shape, dtype)
            got = []
            for plain in (True, False):
                tensors = {n: Stub(*spec[n]) for n in names}
                got.append(_outcome(rope, monkeypatch, tensors, inplace, plain))
            assert got[0] == got[1] != "unexpected", (change, names, inplace, got)
            seen.add(got[0] == "accepted")
    assert seen == {True, False}


@pytest.mark.parametrize("name", list(USUAL))
@pytest.mark.parametrize("change", [{"device": "cpu"}, {"device": "cuda:1"}, {"contiguous": False}])
def test_plain_devices_and_layouts(rope, monkeypatch, name, change):
    for inplace in (False, True):
        got = []
        for plain in (True, False):
            tensors = {n: Stub(*USUAL[n], **(change if n == name else {})) for n in USUAL}
            got.append(_outcome(rope, monkeypatch, tensors, inplace, plain))
        assert got[0] == got[1] != "unexpected"
