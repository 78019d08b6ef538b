"""The share of the device memory that formal solutions keep intensity cubes in
(adjoint._kept_cubes), with the allocator's figures set by the test: CPU tensors stand for
the cubes, one byte a unit."""
import threading

import numpy as np
import pytest
import torch

from dispatch_amd import adjoint


class Memory:
    """A device of `total` bytes: `used` held by the process, cubes among it, `others` by others."""

    def __init__(self, monkeypatch, total, used=0, others=0, cached=0):
        self.total, self.used, self.others, self.cached = total, used, others, cached
        monkeypatch.setattr(torch.cuda, "memory_allocated", lambda d: self.used + kept())
        monkeypatch.setattr(torch.cuda, "memory_reserved", lambda d: self.used + kept() + self.cached)
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d: (
            self.total - self.others - self.used - kept() - self.cached, self.total))


def kept():
    return sum(c.held(torch.device("cpu")) for c in list(adjoint._live.values()))


def solution(cube, nray):
    """What the forward of one solution keeps."""
    c = adjoint._Cubes()
    for r in range(adjoint._kept_cubes(cube, nray)):
        c.add(r, cube)
    return c


@pytest.fixture(autouse=True)
def nothing_else_kept():
    adjoint._give_back(torch.device("cpu"))


@pytest.mark.parametrize("cached", [0, 300])
def test_half_of_what_the_backward_pass_leaves(monkeypatch, cached):
    cube = torch.zeros(10, dtype=torch.uint8)
    m = Memory(monkeypatch, 1000, used=100, others=70, cached=cached)
    # 1000 - 100 - 70 free, 30 for the backward pass, 100 for the caller's: 700, half 350
    assert adjoint._kept_cubes(cube, 100) == 35
    assert adjoint._kept_cubes(cube, 12) == 12
    m.used = 430
    assert adjoint._kept_cubes(cube, 12) == 2
    m.used = 460
    assert adjoint._kept_cubes(cube, 12) == 0


def test_many_solutions_share_the_half_and_give_it_back(monkeypatch):
    """Windows of one graph: each solution's chi and S stay, its cubes are kept beside the
    earlier ones'; all cubes together stay within the half, and are gone when the rest
    holds half of the device."""
    cube = torch.zeros(10, dtype=torch.uint8)
    m = Memory(monkeypatch, 2000)
    waiting, most = [], []
    while m.used + 30 < 1000:
        m.used += 20
        waiting.append(solution(cube, 12))
        room = (2000 - 2 * m.used - 30) // 2
        assert kept() <= max(0, room)
        most.append(kept())
    assert max(most) > 600 and kept() == 0
    assert all(not c.by_ray for c in waiting[:-1])


def test_cubes_go_with_their_graph_and_by_thread(monkeypatch):
    cube = torch.zeros(10, dtype=torch.uint8)
    Memory(monkeypatch, 10000)
    a, b = solution(cube, 4), solution(cube, 4)
    assert kept() == 80
    del a
    assert kept() == 40
    mine = b.pop(0)
    t = threading.Thread(target=adjoint._give_back, args=(torch.device("cpu"),))
    t.start()
    t.join()
    assert kept() == 0 and b.pop(1) is None and mine.numel() == 10


def test_allocations_come_before_cubes(monkeypatch):
    cube = torch.zeros(10, dtype=torch.uint8)
    Memory(monkeypatch, 10000)
    s = solution(cube, 4)
    asked = []

    def make():
        asked.append(kept())
        if kept():
            raise torch.OutOfMemoryError("no room beside the cubes")
        return 7

    assert adjoint._alloc(torch.device("cpu"), make) == 7 and asked == [40, 0] and not s.by_ray

    def never():
        raise torch.OutOfMemoryError("no room at all")

    with pytest.raises(torch.OutOfMemoryError):
        adjoint._alloc(torch.device("cpu"), never)
    monkeypatch.setattr(torch, "empty_like", lambda t: never())
    assert s.add(0, cube) is None and not s.by_ray


@pytest.mark.parametrize("keep", [-1, "all", 1.5])
def test_keep_is_a_number_or_auto(keep):
    with pytest.raises(ValueError, match="keep"):
        adjoint.RaySet(None, np.zeros((1, 3)), np.ones(1), (1, 1, 1), None, [], None, None, keep=keep)
