"""What the plan cache (bpt_amd/plan.py) tells the native host path, whose table answers calls by the addresses of their index tensors:
an entry is let in only while its plans are in the cache, and a plan that other threads may have taken from the cache is not
replaced.  CPU only: the native side is a stub, other threads' doings are put where they would fall."""
import os
import subprocess
import sys

import pytest
import torch

from bpt_amd import plan as plan_mod


class Native:
    """Keeps the rules of bptop.so's table: entries by key, dropped with any of their plans."""

    def __init__(self):
        self.table = {}

    def remember(self, generation, kind, index, extra, a, b, plans):
        self.table[kind, tuple(id(t) for t in index)] = plans

    def forget(self, plan):
        self.table = {k: ps for k, ps in self.table.items() if not any(p is plan for p in ps)}

    def clear(self):
        self.table = {}

    def take_used(self):
        return []


class FakePlan:
    def __init__(self, *args, groups=None):
        pass

    def device_bytes(self):
        return 1


def side(n=3):
    return tuple(torch.arange(n) for _ in range(4))


@pytest.fixture
def cache(monkeypatch):
    monkeypatch.setattr(plan_mod, "Plan", FakePlan)
    c = plan_mod.PlanCache(capacity=4)
    c.native = Native()
    return c


def choice(index):
    return 0, 0, list(index), [0] * 6, 1, 0


def test_a_plan_in_the_cache_is_remembered(cache):
    a, b = side(), side()
    pa, pb = cache.get(*a, 3, 3), cache.get(*b, 3, 3)
    cache.remember((pa, pb), *choice(a + b))
    assert list(cache.native.table.values()) == [(pa, pb)]


@pytest.mark.parametrize("gone", [0, 1])
def test_a_plan_dropped_since_it_was_asked_for_is_not_remembered(cache, gone):
    sides = side(), side()
    plans = [cache.get(*s, 3, 3) for s in sides]
    if gone == 0:                                    # (the other one was used since)
        cache.get(*sides[1], 3, 3)
    else:
        cache.get(*sides[0], 3, 3)
    for _ in range(3):                               # another thread's graphs
        cache.get(*side(), 3, 3)
    assert [any(p is q for q, _ in cache._d.values()) for p in plans] == [gone != 0, gone != 1]
    cache.remember(tuple(plans), *choice(sides[0] + sides[1]))
    assert not cache.native.table


def test_a_cleared_cache_remembers_nothing_of_before(cache):
    a = side()
    pa = cache.get(*a, 3, 3)
    cache.clear()
    cache.remember((pa,), *choice(a))
    assert not cache.native.table


def test_entries_go_with_their_plans(cache):
    a = side()
    cache.remember((cache.get(*a, 3, 3),), *choice(a))
    for _ in range(4):
        cache.get(*side(), 3, 3)
    assert not cache.native.table


def test_two_threads_that_build_the_same_plan_share_the_first(cache, monkeypatch):
    a, meanwhile = side(), []

    class Slow(FakePlan):                            # while this one is built, another thread asks, builds and gets its own
        def __init__(self, *args, groups=None):
            if not meanwhile:
                monkeypatch.setattr(plan_mod, "Plan", FakePlan)
                meanwhile.append(cache.get(*a, 3, 3))
                cache.remember((meanwhile[0],), *choice(a))

    monkeypatch.setattr(plan_mod, "Plan", Slow)
    mine = cache.get(*a, 3, 3)
    assert mine is meanwhile[0] and len(cache._d) == 1 and cache._total == 1
    cache.remember((mine,), *choice(a))
    for _ in range(4):
        cache.get(*side(), 3, 3)
    assert not any(p is mine for p, _ in cache._d.values()) and not cache.native.table


def test_two_threads_that_build_both_sides_share_the_first(cache, monkeypatch):
    class Index:                                     # (plans of both sides are built together on the GPU only)
        device, is_cuda, _version = "cuda:0", True, 0

        def data_ptr(self):
            return id(self)

        def numel(self):
            return 3

    sides = [(*(Index() for _ in range(4)), 3, 3, 64, None) for _ in range(2)]
    built = []

    def tile_plans(sides_):
        mine = [FakePlan(), FakePlan()]
        built.append(mine)
        if len(built) == 1:
            cache.put_tile_plans(sides)              # the other thread, from beginning to end
        return mine

    monkeypatch.setattr(plan_mod.DevicePlan, "tile_plans", staticmethod(tile_plans))
    cache.put_tile_plans(sides)
    assert len(built) == 2 and [p for p, _ in cache._d.values()] == built[1] and cache._total == 2


def test_joint_plans_without_the_ops():
    """DevicePlan.tile_plans where nothing has imported the ops: tensors that are not on a GPU are left to the other builders."""
    code = ("import sys, torch; from bpt_amd.plan import DevicePlan; t = torch.zeros(2, dtype=torch.int64); "
            "assert 'bpt_amd.graphop' not in sys.modules; assert DevicePlan.tile_plans([(t[:1], t, t[:1], t[:1], 1, 1, 64, None)]) is None")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    subprocess.run([sys.executable, "-c", code], cwd=root, check=True)
