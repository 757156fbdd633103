"""What was launched stays listed until a wait for it is over: a second wait, of another thread or inside the block of
``syncing``, does not return before the device is done, and no launch is lost between the two."""

import threading

import pytest
import torch

from odc_amd import ReductionService
from odc_amd.primitives import scatter_accumulate, utils


class Stream:
    """A stream whose work is done once `done` is set."""

    def __init__(self, handle):
        self.cuda_stream, self.done, self.waited, self.asked = handle, threading.Event(), 0, threading.Event()

    def synchronize(self):
        self.asked.set()
        assert self.done.wait(20)
        self.waited += 1

    def wait_event(self, event):
        pass


class Event:
    def record(self, stream):
        self.stream = stream

    def synchronize(self):
        self.stream.synchronize()


@pytest.fixture
def streams(monkeypatch, launch_list):
    """Two streams with launches, 1 (the current one) and 2; wrapped as the services leave them."""
    made = {1: Stream(1), 2: Stream(2)}
    launch_list.update({1: None, 2: made[2]})
    monkeypatch.setattr(utils, "stream_from_handle", made.__getitem__)
    for module in (utils, scatter_accumulate):
        monkeypatch.setattr(module, "get_world", lambda: type("World", (), {"device": 0}))
    monkeypatch.setattr(scatter_accumulate, "_is_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: made[1])
    monkeypatch.setattr(torch.cuda, "Event", Event)
    return made


def _in_thread(call):
    thread = threading.Thread(target=call, daemon=True)
    thread.start()
    return thread


def _release(streams):
    for s in streams.values():
        s.done.set()


def test_a_second_wait_does_not_return_early(streams):
    first = _in_thread(utils.wait_for_launches)
    assert streams[1].asked.wait(20)
    second = _in_thread(ReductionService().sync)
    second.join(0.3)
    assert second.is_alive(), "returned with launches in flight"
    _release(streams)
    first.join(20), second.join(20)
    assert not first.is_alive() and not second.is_alive()
    assert all(s.waited == 2 for s in streams.values())
    utils.wait_for_launches()  # nothing is listed any more
    assert all(s.waited == 2 for s in streams.values())


@pytest.mark.parametrize("inside", [False, True], ids=["another thread", "the block"])
def test_a_wait_during_the_block_of_syncing(streams, inside):
    service, order = ReductionService(), []

    def minibatch():
        with service.syncing():
            if inside:
                service.sync()
                order.append("inside")
            else:
                other = _in_thread(service.sync)
                other.join(0.3)
                order.append(other.is_alive())
                _release(streams)
                other.join(20)
                order.append(other.is_alive())

    thread = _in_thread(minibatch)
    if inside:
        thread.join(0.3)
        assert order == [], "returned with launches in flight"
        _release(streams)
    thread.join(20)
    assert not thread.is_alive() and order == (["inside"] if inside else [True, False])
    assert all(s.waited == 2 for s in streams.values())


def test_a_launch_behind_a_wait_that_came_between(streams, monkeypatch):
    """Another thread waits just as this one is about to launch: what is launched then is still listed."""
    _release(streams)
    service = ReductionService()
    monkeypatch.setattr(service, "_order_after_writers", lambda keys, stream: None)
    world = type("World", (), {"device": 0, "arena": type("Arena", (), {"raw_handle": 0})})
    monkeypatch.setattr(scatter_accumulate, "get_world", lambda: world)
    monkeypatch.setattr(utils, "_current_raw_stream", lambda device: 1)

    class Items:
        grad_code = acc_code = 0

        def launch(self, arena, stream, store):
            utils.wait_for_launches()
            streams[1].done.clear()
            return 0

    service._launch(("k",), Items(), 1, 0, 0, False)
    waiting = _in_thread(service.sync)
    waiting.join(0.3)
    assert waiting.is_alive(), "returned with a launch in flight"
    _release(streams)
    waiting.join(20)
    assert not waiting.is_alive()


def test_a_wait_that_fails_loses_nothing(streams):
    """(under capture, for one)"""
    def refuse():
        raise ValueError("not now")

    def block():
        with ReductionService().syncing():
            pass

    for wait in (utils.wait_for_launches, lambda: ReductionService().sync(), block):
        streams[2].synchronize = refuse
        _release(streams)
        with pytest.raises(ValueError):
            wait()
        del streams[2].synchronize
        waited = streams[2].waited
        utils.wait_for_launches()
        assert streams[2].waited == waited + 1
        utils._launch_streams[2] = streams[2]


@pytest.mark.parametrize("refused", [False, True])
def test_the_block_under_capture(streams, monkeypatch, refused):
    """As sync does: it waits for streams that may be waited for, and is refused for the captured one."""
    monkeypatch.setattr(scatter_accumulate, "_is_capturing", lambda: True)
    service, ran = ReductionService(), []
    service.dispatched_tasks = 3

    def no_events(*_):
        raise AssertionError("recorded an event into the graph")

    def refuse():
        raise ValueError("capturing")

    monkeypatch.setattr(Event, "record", no_events)
    _release(streams)
    if refused:
        streams[1].synchronize = refuse
        with pytest.raises(ValueError):
            with service.syncing():
                ran.append(True)
        assert not ran and service.dispatched_tasks == 3 and set(utils._launch_streams) == {1, 2}
        return
    with service.syncing():
        ran.append(service.dispatched_tasks)
    assert ran == [0] and not utils._launch_streams and not utils._waits


def test_the_current_stream_stays_listed(streams):
    """It has the launches of the block, as a rule: a sync behind the block waits for it again, and for no other."""
    _release(streams)
    with ReductionService().syncing():
        assert set(utils._launch_streams) == {1}
    assert set(utils._launch_streams) == {1} and not utils._waits
    utils.wait_for_launches()
    assert streams[1].waited == 2 and streams[2].waited == 1 and not utils._launch_streams


def test_an_order_that_fails_loses_nothing(streams, monkeypatch):
    def refuse(*_):
        raise ValueError("not now")

    monkeypatch.setattr(Event, "record", refuse)
    with pytest.raises(ValueError):
        with ReductionService().syncing():
            raise AssertionError("the block ran")
    assert set(utils._launch_streams) == {1, 2} and not utils._waits


def test_tasks_dispatched_during_a_wait_stay_counted(streams):
    for wait in ("sync", "syncing"):
        service = ReductionService()
        service.dispatched_tasks = 5
        utils._launch_streams[2] = streams[2]
        _release(streams)
        original = streams[2].synchronize

        def synchronize():
            service.dispatched_tasks += 2  # another thread's
            original()

        streams[2].synchronize = synchronize
        if wait == "sync":
            service.sync()
        else:
            with service.syncing():
                pass
        del streams[2].synchronize
        assert service.dispatched_tasks == 2
        service.sync()
        assert service.dispatched_tasks == 0


def test_a_count_that_is_set_during_a_wait(streams):
    service = ReductionService()
    service.dispatched_tasks = 5
    _release(streams)
    with service.syncing():
        service.dispatched_tasks = 0
        assert service.dispatched_tasks == 0
        service.dispatched_tasks += 2
    assert service.dispatched_tasks == 2
    service.sync()
    assert service.dispatched_tasks == 0
