"""The recorded decode runner's waits, on the CPU: streams are queues of what was enqueued on them and run only when
something waits for them, so a wait that is missing shows as the numbers of before."""
import threading
import time
from types import SimpleNamespace

import pytest
import torch

from llm_infer_amd.engine import decode
from llm_infer_amd.kernels import ops


class Stream:
    def __init__(self):
        self.queue = []

    def run(self):
        while self.queue:
            self.queue.pop(0)()

    synchronize = run

    def wait_stream(self, other):
        self.queue.append(other.run)

    def query(self):
        return not self.queue


class Buffer:
    """Numbers on the device: what is copied into them or out of them is enqueued on the current stream."""

    def __init__(self, device, values, n=None):
        self.device, self.values, self.n = device, values, n

    def __getitem__(self, part):
        return Buffer(self.device, self.values, part.stop)

    def copy_(self, src, non_blocking=False):
        if isinstance(src, Buffer):
            self.device.current.queue.append(lambda: self.values.__setitem__(slice(0, self.n), src.values[:src.n]))
        else:
            numbers = src.tolist()
            self.device.current.queue.append(lambda: self.values.__setitem__(slice(0, self.n), numbers))

    def fill_(self, v):
        self.device.current.queue.append(lambda: self.values.__setitem__(slice(0, len(self.values)), [v] * len(self.values)))

    def tolist(self):
        return list(self.values[:self.n])


class Graphs(dict):
    """An engine's recorded steps: none is ever kept, so every step runs eagerly."""

    def __setitem__(self, key, entry):
        pass


class Device:
    """Two streams and an engine whose step adds the slot's number to each row's token."""

    def __init__(self, monkeypatch, n_slots=4):
        self.a, self.b = Stream(), Stream()
        self.current, self.ring, self.fails = self.a, {}, 0
        monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: self.current)
        monkeypatch.setattr(torch.cuda, "stream", self.on)
        monkeypatch.setattr(decode.Tensor, "pinned", staticmethod(lambda shape, dtype: torch.zeros(shape, dtype=dtype)))
        monkeypatch.setattr(ops, "wait_tokens", self.wait_tokens)
        cache = SimpleNamespace(n_slots=n_slots, scratch_slot=n_slots, lens=[5] * n_slots, lens_dev=None, grow=self.grow,
                                trim_windows=lambda slots: None)
        self.engine = SimpleNamespace(cache=cache, device="cpu", model=SimpleNamespace(positions={}), _graphs=Graphs(), _graph_bufs=None,
                                      decode_counts={"eager": 0, "recorded": 0, "replayed": 0})

    def grow(self, slots, lens, sync_lens):
        for s, n in zip(slots, lens):
            self.engine.cache.lens[s] = n

    def on(self, stream):
        from contextlib import contextmanager

        @contextmanager
        def inside():
            before, self.current = self.current, stream
            yield
            self.current = before
        return inside()

    def runner(self):
        runner = decode.GraphDecodeRunner(self.engine, SimpleNamespace(temperature=0.0))
        b = runner.bufs
        if not isinstance(b["tokens"], Buffer):
            for name in ("tokens", "slots", "steps"):
                b[name] = Buffer(self, [0] * self.engine.cache.n_slots)
            b["host"][1] = Buffer(self, [0] * self.engine.cache.n_slots)

        def body(n, bucket, pages):
            def prepare():
                number = b["steps"].values[0] + 1
                b["steps"].values[:] = [number] * len(b["steps"].values)
                self.ring[number] = list(b["tokens"].values)

            def rest():
                b["tokens"].values[:n] = [t + s + 1 for t, s in zip(b["tokens"].values[:n], b["slots"].values[:n])]

            self.current.queue.append(prepare)
            if self.fails:
                self.fails -= 1
                raise RuntimeError("this step fails")
            self.current.queue.append(rest)
        runner._body = body
        return runner

    def wait_tokens(self, ring, n, step, stream=None):
        """The device goes on by itself while the host polls; a stream that is done without the step's tokens is an error."""
        queue = (stream or self.current).queue
        while step not in self.ring:
            if not queue:
                raise ops.KernelError("the device is done")
            queue.pop(0)()
        return self.ring[step][:n]


def test_a_step_is_waited_for_on_its_own_stream(monkeypatch):
    """Steps launched ahead under one stream, collected or dropped under another."""
    dev = Device(monkeypatch)
    runner = dev.runner()
    assert runner.run([0, 2], [10, 20], may_follow=True) == [11, 23]
    dev.current = dev.b
    assert runner.run([0, 2], [11, 23]) == [12, 26]                      # the one ahead, from its own stream
    assert runner.run([0, 2], [12, 26], may_follow=True) == [13, 29]
    dev.current = dev.a
    assert runner.run([0, 2], [13, 29], may_follow=True) == [14, 32]     # the next one behind it, on this stream
    dev.current = dev.b
    assert not dev.a.query()
    runner.drain()
    assert dev.a.query()                                                 # nothing is left that works on the slots


def test_runners_of_one_engine_keep_their_own_tokens(monkeypatch):
    """Another runner's step, for other sequences, more of them or the same, between a step that was enqueued ahead and the call that
    asks for its tokens; and tokens that are not those of the step before."""
    dev = Device(monkeypatch)
    one, two = dev.runner(), dev.runner()
    assert one.run([0, 2], [10, 20], may_follow=True) == [11, 23]
    assert two.run([1], [50], may_follow=True) == [52]
    assert one.run([0, 2], [11, 23]) == [12, 26]                         # the one that was ahead of the other runner's
    assert one.run([0, 2], [12, 26], may_follow=True) == [13, 29]
    assert two.run([1], [52], may_follow=True) == [54]                   # likewise: and none is enqueued behind it
    assert two.run([1], [54], may_follow=True) == [56]
    assert one.run([0, 2], [13, 29], may_follow=True) == [14, 32]
    assert two.run([1], [56]) == [58]
    one.drain()
    assert two.run([0, 2], [70, 80]) == [71, 83]
    assert one.run([0, 2], [90, 40]) == [91, 43]                         # the same sequences, not the tokens that lie there
    got = one.run([0, 2], [91, 43])
    got[0] = 7
    assert one.run([0, 2], got) == [8, 49]


@pytest.mark.parametrize("fails", [1, 2])
def test_a_step_that_fails_says_why_and_the_next_ones_are_right(monkeypatch, fails):
    """An error while a step is being enqueued reaches the caller as it is, whatever state the device is in, and no later step is taken
    for the one that failed, whose first kernel may have run."""
    dev = Device(monkeypatch)
    runner = dev.runner()
    assert runner.run([0, 2], [10, 20], may_follow=True) == [11, 23]
    fill, lost = Buffer.fill_, lambda self, v: (_ for _ in ()).throw(ValueError("the device is lost"))
    dev.fails = 1
    monkeypatch.setattr(Buffer, "fill_", lost)
    with pytest.raises(RuntimeError, match="this step fails"):
        runner.run([0, 2], [11, 23], may_follow=True)                    # (fails as the one behind it is enqueued)
    monkeypatch.setattr(Buffer, "fill_", fill)
    dev.fails = fails - 1
    for _ in range(fails - 1):
        with pytest.raises(RuntimeError, match="this step fails"):
            runner.run([0, 2], [30, 40])
    assert runner.run([0, 2], [30, 40], may_follow=True) == [31, 43]
    assert runner.run([0, 2], [31, 43], may_follow=True) == [32, 46]
    assert runner.run([0, 2], [32, 46]) == [33, 49]
    assert runner.run([1], [5], may_follow=True) == [7]
    runner.drain()


def test_a_step_ahead_outlives_another_runners_failure(monkeypatch):
    """Another runner's step that fails on the host, as one that the cache has no room for does, takes nothing from a step enqueued ahead:
    its tokens are its own, and not those of the step that is then enqueued behind it under a number that is not the next."""
    dev = Device(monkeypatch)
    one, two = dev.runner(), dev.runner()
    assert one.run([0, 2], [10, 20], may_follow=True) == [11, 23]
    grow = dev.engine.cache.grow
    dev.engine.cache.grow = lambda *args, **kw: (_ for _ in ()).throw(RuntimeError("no room"))
    with pytest.raises(RuntimeError, match="no room"):
        two.run([1], [50])
    dev.engine.cache.grow = grow
    assert one.run([0, 2], [11, 23], may_follow=True) == [12, 26]
    assert one.run([0, 2], [12, 26]) == [13, 29]
    assert two.run([1], [50]) == [52]


def test_tokens_that_are_waited_for_come_from_the_steps_own_stream(monkeypatch):
    """Another stream that is idle says nothing about the step's: no error while that one still runs."""
    idle, busy = SimpleNamespace(query=lambda: True), SimpleNamespace(query=lambda: False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: idle)
    ring = torch.zeros((ops.TOKEN_RING, 2), dtype=torch.int64)

    def later():
        time.sleep(1.3)
        ring[3, 0], ring[3, 1] = 7 << 32 | 40, 7 << 32 | 41
    writer = threading.Thread(target=later)
    writer.start()
    try:
        assert ops.wait_tokens(ring, 2, 7, busy) == [40, 41]
    finally:
        writer.join()
    with pytest.raises(ops.KernelError):
        ops.wait_tokens(ring, 2, 8)
