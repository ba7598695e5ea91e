"""The differentiable NUFFT's plan pool (gadgetron_amd/autograd.py) with stand-in plans
and trajectories in host memory: which plans are made, which are taken again, and
which are let go.
"""
import gc

import pytest
import torch

from gadgetron_amd import autograd as ag

STREAM = 17


class Plan:
    made = []

    def __init__(self, N, Nos, W, os_factor):
        self.N = tuple(N)
        Plan.made.append(self.N)

    def preprocess(self, k, stream):
        pass


@pytest.fixture(autouse=True)
def pool(monkeypatch):
    monkeypatch.setattr(ag, "NFFTPlan", Plan)
    ag.clear_plan_cache()
    gc.collect()
    ag.clear_plan_cache()
    Plan.made.clear()
    yield
    ag.clear_plan_cache()


def step(N, stream=STREAM):
    """One optimiser step: a new trajectory, its lease let go at the end."""
    k = torch.rand(1, 8, 2)
    lease = ag._plan_for(k, N, 5.5, 1.5, stream)
    assert lease.plan.N == tuple(N)
    return lease.plan


def test_steps_of_one_size_share_two_plans():
    # the cache entry of the last trajectory holds its plan until the next one is looked up
    for _ in range(6):
        step((32, 32))
    assert len(Plan.made) <= 2


def test_sizes_no_longer_used_give_way():
    for N in ((32, 32), (48, 48), (64, 64), (80, 80)):
        for _ in range(6):
            step(N)
        assert Plan.made.count(N) <= 2
    assert len(ag._POOL) <= ag.PLAN_POOL_SIZE


def test_the_longest_unused_plan_goes_first():
    plans = [step((n, n)) for n in (32, 48, 64, 80)]
    ag._PLANS.clear()  # the leases end in this order
    assert [e[1] for e in ag._POOL] == plans[-ag.PLAN_POOL_SIZE:]
    assert ag._take(ag._POOL[1][0]) is plans[-1]
    assert [e[1] for e in ag._POOL] == [plans[-2]]


def test_a_live_lease_keeps_its_plan():
    k = torch.rand(1, 8, 2)
    lease = ag._plan_for(k, (32, 32), 5.5, 1.5, STREAM)
    others = {id(step((32, 32))) for _ in range(4)}
    assert id(lease.plan) not in others


def test_another_stream_does_not_take_a_pooled_plan():
    first = step((32, 32))
    ag._PLANS.clear()
    assert [e[1] for e in ag._POOL] == [first]
    assert step((32, 32), stream=STREAM + 1) is not first
    assert first in [e[1] for e in ag._POOL]
    assert step((32, 32)) is first


def test_a_plan_used_on_two_streams_is_not_pooled():
    k = torch.rand(1, 8, 2)
    lease = ag._plan_for(k, (32, 32), 5.5, 1.5, STREAM)
    assert ag._plan_for(k, (32, 32), 5.5, 1.5, STREAM + 1) is lease
    del lease
    ag._PLANS.clear()
    assert not ag._POOL
