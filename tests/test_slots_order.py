"""The pinned slots' order of copies and waits, on a model of asynchronous copies (CPU): a copy between a
slot and a device tensor waits in the queue of that tensor's device and is made when something waits for
the queue.  What the host reads before that is what the slot held before."""
import collections

import pytest
import torch

from holodeck_amd import device as D

SLOT = 4 << 10


class Sim(torch.Tensor):
    """A tensor with a place of its own: 'slot', or a device index."""
    place = None

    @classmethod
    def at(cls, t, place):
        t = t.as_subclass(cls)
        t.place = place
        return t

    @property
    def device(self):
        return torch.device("cuda", self.place) if isinstance(self.place, int) else torch.device("cpu")

    def __getitem__(self, k):
        return Sim.at(self.as_subclass(torch.Tensor)[k], self.place)

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        if func is not torch.Tensor.copy_:
            return super().__torch_function__(func, types, args, kwargs or {})
        dst, src = args
        place = [t.place for t in (dst, src) if isinstance(t, Sim) and isinstance(t.place, int)]
        d, s = dst.as_subclass(torch.Tensor), src.as_subclass(torch.Tensor)
        if place:
            assert kwargs == {"non_blocking": True}
            World.queue[place[0]].append(lambda: d.copy_(s))
        else:
            d.copy_(s)
        return dst


class World:
    """One stream per device; device 0 is the current one."""
    queue = collections.defaultdict(list)
    interrupt = 0      # raise at this wait (1: the first)

    @classmethod
    def drain(cls, place, upto=None):
        q = cls.queue[place]
        while q and (upto is None or upto > 0):
            q.pop(0)()
            upto = None if upto is None else upto - 1

    class Stream:
        def __init__(self, place):
            self.place = place

        def synchronize(self):
            World.drain(self.place)

    class Event:
        def record(self, stream=None):
            self.place = 0 if stream is None else stream.place
            self.upto = list(World.queue[self.place])

        def synchronize(self):
            World.interrupt -= 1
            if World.interrupt == 0:
                raise KeyboardInterrupt
            for op in self.upto:
                if op in World.queue[self.place]:
                    World.queue[self.place].remove(op)
                    op()


@pytest.fixture
def slots(monkeypatch):
    World.queue.clear()
    World.interrupt = 0
    real_empty = torch.empty

    def empty(*shape, **kw):
        if not kw.pop("pin_memory", False):
            return real_empty(*shape, **kw)
        return Sim.at(real_empty(*shape, **kw).fill_(255), "slot")

    def current_stream(device=None):
        index = getattr(device, "index", device)
        return World.Stream(0 if index is None else index)

    monkeypatch.setattr(torch, "empty", empty)
    monkeypatch.setattr(torch.cuda, "Event", World.Event)
    monkeypatch.setattr(torch.cuda, "current_stream", current_stream)
    monkeypatch.setattr(D, "SLOT_BYTES", SLOT)
    return D._Slots()


def _data(n, seed):
    return torch.randint(0, 200, (n,), dtype=torch.uint8, generator=torch.Generator().manual_seed(seed))


@pytest.mark.parametrize("place", [0, 1])
@pytest.mark.parametrize("n", [1, SLOT - 1, SLOT, SLOT + 1, 5 * SLOT + 7])
def test_copies_wait_for_the_tensors_own_device(slots, place, n):
    a = _data(n, n)
    got = torch.zeros(n, dtype=torch.uint8)
    assert slots.fetch(Sim.at(a.clone(), place), got)
    assert torch.equal(got, a)
    put = torch.zeros(n, dtype=torch.uint8)
    assert slots.push(a.clone(), Sim.at(put, place))
    assert torch.equal(put, a)


@pytest.mark.parametrize("way", ["fetch", "push"])
@pytest.mark.parametrize("wait", [1, 2])
def test_an_interrupted_copy_keeps_its_slots_to_itself(slots, way, wait):
    """The copies still in flight when a wait is interrupted run after the next caller has filled its slots."""
    a, b = _data(6 * SLOT, 1), _data(2 * SLOT, 2)
    put = torch.zeros_like(a)
    World.interrupt = wait
    with pytest.raises(KeyboardInterrupt):
        if way == "fetch":
            slots.fetch(Sim.at(a.clone(), 1), torch.zeros_like(a))
        else:
            slots.push(a.clone(), Sim.at(put, 1))
    late = list(World.queue[1])
    assert late
    World.queue[1].clear()
    World.interrupt = 0
    got = torch.zeros_like(b)
    land = D._Slots._land

    def after_the_late_ones(dst, slot, ev):
        ev.synchronize()
        while late:
            late.pop(0)()
        dst.copy_(slot)

    slots._land = after_the_late_ones if way == "fetch" else land
    assert slots.fetch(Sim.at(b.clone(), 0), got)
    assert torch.equal(got, b)
    if way == "push":      # what was queued before the interruption still holds its own data
        n = len(late)
        while late:
            late.pop(0)()
        done = [k for k in range(6) if put[k * SLOT:(k + 1) * SLOT].any()]
        assert len(done) >= n
        for k in done:
            assert torch.equal(put[k * SLOT:(k + 1) * SLOT], a[k * SLOT:(k + 1) * SLOT])


def test_without_pinned_memory_the_runtime_copies(slots, monkeypatch):
    """No pinned memory to be had: the caller is told to take the runtime's own copy, each time."""
    def none_left(*shape, **kw):
        raise torch.cuda.OutOfMemoryError("HIP out of memory")
    monkeypatch.setattr(torch, "empty", none_left)
    a = _data(9, 3)
    for _ in range(2):
        assert not slots.fetch(Sim.at(a.clone(), 0), a) and not slots.push(a, Sim.at(a.clone(), 0))
