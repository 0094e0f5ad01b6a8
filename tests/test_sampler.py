"""What the sampler keeps on the host between a step and its result, with stand-ins for the device's events."""
import threading
import weakref

import pytest
import torch

from litinfer_amd.sampling import Sampler, sampler


class Event:
    def __init__(self, done=False, wait=None):
        self.done, self.wait = done, wait

    def query(self):
        if self.wait is not None:
            self.wait()
        return self.done


@pytest.fixture(autouse=True)
def nothing_unread(monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)      # (there is no device to ask here)
    sampler._unread.clear()
    yield
    sampler._unread.clear()


def _let_go(event, by_kernel=True):
    host = torch.empty(4, dtype=torch.int32)
    seen = weakref.ref(host)
    sampler.PendingTokens(Sampler("cpu"), host, 4, event, by_kernel=by_kernel)
    del host
    return seen


def test_memory_of_an_unread_result_stays_until_the_device_has_written_it():
    first, second = Event(), Event()
    a, b = _let_go(first), _let_go(second)
    smp = Sampler("cpu")
    smp._host_buffer(4)
    assert a() is not None and b() is not None
    second.done = True
    smp._host_buffer(4)                                    # (the entry at the head has not come: the one behind it goes all the same)
    assert a() is not None and b() is None
    first.done = True
    smp._host_buffer(4)
    assert a() is None and not sampler._unread


def test_two_threads_never_drop_an_entry_that_was_not_asked():
    both = threading.Barrier(2)

    def meet():                                            # (until the other thread is here too, or is known not to come)
        try:
            both.wait(timeout=0.5)
        except threading.BrokenBarrierError:
            pass
    kept = []
    for _ in range(3):
        both.reset()
        _let_go(Event(done=True, wait=meet))
        kept.append(_let_go(Event(done=False)))
        threads = [threading.Thread(target=sampler._drain) for _ in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert all(k() is not None for k in kept)


def test_an_event_that_cannot_be_asked_keeps_its_entry():
    def broken():
        raise RuntimeError("no answer")
    a = _let_go(Event(wait=broken))
    with pytest.raises(RuntimeError):
        sampler._drain()
    assert a() is not None and not sampler._unread_lock.locked()


def test_a_recording_asks_no_event(monkeypatch):
    a = _let_go(Event(done=True))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    Sampler("cpu")._host_buffer(4)
    assert a() is not None
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    Sampler("cpu")._host_buffer(4)
    assert a() is None


def test_results_that_are_let_go_do_not_pile_up():
    smp = Sampler("cpu")
    for i in range(1000):
        smp._host_buffer(4)
        assert _let_go(Event(done=True), by_kernel=i % 2 == 0)() is None or i % 2 == 0
        assert len(sampler._unread) <= 1
    for _ in range(200):                                   # a device that stands still for a while
        _let_go(Event(done=False))
    for entry in sampler._unread:
        entry[0].done = True
    for _ in range(26):
        smp._host_buffer(4)
    assert not sampler._unread


def test_written_memory_of_an_unread_result_serves_the_next_call():
    smp, event = Sampler("cpu"), Event()
    seen = _let_go(event)
    assert smp._host_buffer(4) is not seen()               # (still to be written)
    event.done = True
    assert smp._host_buffer(5) is not seen() and not sampler._unread       # (too short: it goes)
    seen = _let_go(Event(done=True))
    got = smp._host_buffer(4)
    assert got is seen() and smp._host_buffer(4) is not got


def test_an_event_is_recorded_again_only_after_it_was_waited_for(monkeypatch):
    recorded, smp = [], Sampler("cpu")

    def record(ev=None):
        if ev is not None and ev.wait is not None:
            ev.wait()
        recorded.append(ev)
        return ev or Event()
    monkeypatch.setattr(sampler, "record_event", record)
    monkeypatch.setattr(Event, "synchronize", lambda self: setattr(self, "done", True), raising=False)
    first = sampler.PendingTokens(smp, torch.zeros(4, dtype=torch.int32), 4, smp._record())
    own = first._event
    assert smp._record() is not own                        # (nobody has waited for it)
    assert first.result() == first.result() == [0] * 4
    assert smp._record() is own and smp._record() is not own
    assert recorded == [None, None, own, None]

    def other_device():
        raise RuntimeError("an event of another device")
    smp._free_events.append(Event(done=True, wait=other_device))
    assert smp._record().wait is None
    for _ in range(20):
        smp._give_back(torch.zeros(4, dtype=torch.int32), Event(done=True))
    assert len(smp._free_events) <= 8


def test_what_one_kernel_leaves_for_the_next_is_a_thread_s_and_a_stream_s_own(monkeypatch):
    from litinfer_amd.kernels import ops
    cpu, stream = torch.device("cpu"), [1]
    monkeypatch.setattr(ops, "_stream", lambda: stream[0])
    room = ops._Scratch()
    a = room.floats(100, cpu)
    assert room.floats(40, cpu) is a and room.floats(100, cpu) is a
    stream[0] = 2
    b = room.floats(100, cpu)
    assert b.data_ptr() != a.data_ptr()
    other = []
    t = threading.Thread(target=lambda: other.append(room.floats(100, cpu)))
    t.start()
    t.join()
    assert other[0].data_ptr() not in (a.data_ptr(), b.data_ptr())
    stream[0] = 1
    grown = room.floats(101, cpu)
    assert grown.numel() >= 101 and room.floats(100, cpu) is grown and len(room.buffers) == 2
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    own = room.floats(10, cpu)
    assert own is not grown and room.floats(10, cpu) is not own                     # (a recording's replays outlive what is kept here)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    for stream[0] in range(3, 40):
        room.floats(8, cpu)
        assert len(room.buffers) <= room.STREAMS


@pytest.mark.parametrize("name", ["argmax_rows", "sample_rows"])
def test_the_kernels_are_given_room_for_their_rows(monkeypatch, name):
    """The first kernel's part for the second, by the library's own count, whatever sizes came before."""
    from litinfer_amd.kernels import ops
    calls = []
    monkeypatch.setattr(ops, "_gpu", lambda *a: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_run", lambda module, fn, *args: calls.append(args))
    for n, v in ((3, 9000), (64, 151936), (1, 17), (128, 33)):
        x, out = torch.zeros(n, v), torch.zeros(n, dtype=torch.int32)
        if name == "argmax_rows":
            ops.argmax_rows(x, out)
            at = calls[-1][2:4]
            assert at[1] - at[0] == 4 * 32 * n and list(ops._scratch.buffers.values())[0].numel() >= 64 * n
        else:
            f = torch.zeros(n)
            ops.sample_rows(x, f, f.int(), f, f, out)
            assert calls[-1][-1] >= ops._sample_scratch_floats(n, v)
            assert list(ops._scratch.buffers.values())[0].data_ptr() == calls[-1][-2]
    ops._scratch.buffers.clear()
