"""Calls that draw at random or return whole states evaluate their symbolic matrices in
one place, the device, whether their plan is new, reused, or not cached at all: equal
arguments then give equal results.  Checked on the CPU with stand-ins for the device
and the plans."""

import numpy as np
import pytest
import torch

from quantum_amd import plan_cache
from quantum_amd import tfq_simulate_ops as sim


class _Plan:
    workspace_bytes = 256

    def __init__(self, streaming=0):
        self.streaming = streaming
        self.staged = []

    def stats(self):
        raise AssertionError("a call needs one flag, not the counts over all ops")

    def stage_values(self, values):
        self.staged.append(values.copy())

    def set_seed(self, seed):
        self.seed = seed


@pytest.fixture
def fake_device(monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(sim, "_device_and_stream", lambda: (torch.device("cuda", 0), 0))
    plan_cache.clear()
    yield
    plan_cache.set_capacity(8)
    plan_cache.clear()


def _call(values, streaming=0, **kw):
    progs = np.array([b"p"] * len(values), dtype=object)
    return sim._run_cached("op", (progs,), ["a"], values, lambda: _Plan(streaming),
                           lambda plan, where: plan, **kw)


@pytest.mark.parametrize("capacity", [8, 0])
def test_every_call_stages_its_values(fake_device, capacity):
    plan_cache.set_capacity(capacity)
    for k in range(3):
        values = np.full((2, 1), k, np.float32)
        np.testing.assert_array_equal(_call(values, seed=k).staged[-1], values)


def test_plans_that_cannot_be_rebound_keep_the_hosts_matrices(fake_device):
    assert _call(np.ones((2, 1), np.float32), streaming=1).staged == []
    assert _call(np.ones((0, 1), np.float32)).staged == []
