"""What becomes of a stream that its program drops (no GPU: the HIP runtime is the fake of test_runtime_host): its
workspace is freed, its handle serves a later stream, and what its unfinished launches read stays until they are done."""

import gc
import threading
import weakref
from types import SimpleNamespace

import pytest

from krn_amd.dtypes import U8
from krn_amd.runtime import hip, hipapi, library
from tests.test_runtime_host import fake  # noqa: F401


@pytest.fixture
def memory(monkeypatch):
    """Stream-ordered memory: allocation -> (bytes, stream) while it lives, and every free's stream."""
    memory = SimpleNamespace(live={}, freed=[])
    addresses = iter(range(4096, 1 << 60, 4096))

    def malloc_async(nbytes, stream):
        address = next(addresses)
        memory.live[address] = (nbytes, stream)
        return address

    def free_async(pointer, stream):
        memory.freed.append((memory.live.pop(pointer)[1], stream))

    monkeypatch.setattr(hipapi, "malloc_async", malloc_async)
    monkeypatch.setattr(hipapi, "free_async", free_async)
    return memory


@pytest.fixture
def device(fake, memory, monkeypatch):  # noqa: F811
    handles = iter(range(1, 10**6))
    monkeypatch.setattr(hipapi, "device_count", lambda: 1)
    monkeypatch.setattr(hipapi, "keep_pool", lambda ordinal: None)
    monkeypatch.setattr(hipapi, "stream_create", lambda: next(handles))
    monkeypatch.setattr(library, "lib", lambda: None)
    fake.hipSetDevice = lambda ordinal: None
    return hip.HIPDevice("gfx950")


def use(stream, nbytes=1 << 20):
    hip.Launch(SimpleNamespace(name="split"), None)._with_workspace(lambda workspace, handle: None, nbytes)(stream)


def test_a_dropped_idle_stream_gives_back_its_workspace_and_its_handle(device, memory):
    stream = device.stream()
    use(stream)
    stream.sync()
    handle, alive = stream.handle, weakref.ref(stream)
    assert len(memory.live) == 1
    del stream
    assert alive() is None and not memory.live and memory.freed == [(handle, handle)]
    assert device.stream().handle == handle


def test_a_dropped_stream_holds_its_arguments_until_its_work_is_done(device, memory, fake):  # noqa: F811
    stream = device.stream()
    argument = device.empty_on(device.default_stream, U8, 64)
    held = weakref.ref(argument)
    stream.note("k", (argument,))
    handle = stream.handle
    del stream, argument
    gc.collect()
    assert held() is not None
    other = device.stream()  # asks for the first time: an event after the dropped stream's work
    assert held() is not None and other.handle != handle
    another = device.stream()
    assert held() is not None and another.handle not in (handle, other.handle)
    fake.finished.update(fake.recorded)
    assert device.stream().handle == handle and held() is None
    assert memory.freed == [(device.default_stream.handle, device.default_stream.handle)]


def test_a_stream_for_every_request_holds_a_bounded_amount(device, memory, fake):  # noqa: F811
    handles, most = set(), 0
    for _ in range(200):
        with device.stream() as stream:
            use(stream)
            stream.note("k", (device.empty_on(stream, U8, 1 << 20),))
        handles.add(stream.handle)
        fake.finished.update(fake.recorded)  # the device keeps up
        most = max(most, len(memory.live))
    del stream
    assert len(handles) <= 4 and most <= 8
    assert all(made == returned for made, returned in memory.freed)


def test_a_device_sync_covers_dropped_streams(device, memory, fake):  # noqa: F811
    kept, stream = device.stream(), device.stream()
    use(stream)
    idle = device.stream()
    del stream, idle
    before = fake.synced
    device.sync()
    assert fake.synced - before == 4  # the default stream, `kept`, and the two dropped ones
    assert not memory.live and not device._retired and kept is not None


def test_a_stream_dropped_while_a_graph_records_it_is_not_used_again(device, fake, monkeypatch):  # noqa: F811
    recording = set()
    monkeypatch.setattr(hipapi, "capturing", lambda handle: handle in recording)
    forked, empty = device.stream(), device.stream()
    recording |= {forked.handle, empty.handle}
    argument = device.empty_on(device.default_stream, U8, 64)
    held = weakref.ref(argument)
    forked.note("k", (argument,))
    del forked, empty, argument
    assert device.stream().handle not in recording
    recording.clear()  # the recording ends: the graph may be replayed
    fake.finished.update(fake.recorded)
    for _ in range(3):
        device.stream()
        fake.finished.update(fake.recorded)
    assert held() is not None
    device.sync()
    assert held() is None


def test_streams_come_and_go_in_several_threads(device, memory, fake):  # noqa: F811
    failures = []

    def work():
        try:
            for _ in range(200):
                use(device.stream())
                fake.finished.update(list(fake.recorded))
        except Exception as error:  # reported by the assertion below
            failures.append(error)

    threads = [threading.Thread(target=work) for _ in range(4)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    device.sync()
    assert not failures and not memory.live
    assert len(set(device._idle)) == len(device._idle)  # no handle twice


def test_replays_in_flight_hold_the_recording_and_not_the_function(device, monkeypatch):
    """A stream whose replay's function refers to it would otherwise be a cycle through the arguments it holds."""
    monkeypatch.setattr(hip.HIPGraph, "_capture", lambda self, *a, **k: hip.Recording(7, 8, []))
    monkeypatch.setattr(hip, "_release_graph", lambda executable, graph: None)
    stream = device.stream()
    graph = device.graph(lambda: stream)
    monkeypatch.setattr(hipapi.api(), "hipGraphLaunch", lambda executable, handle: None, raising=False)
    with stream:
        graph()
    recording, alive = weakref.ref(graph._recording), weakref.ref(stream)
    del graph, stream
    assert alive() is None and recording() is not None  # held by the dropped stream's unfinished work
    device.sync()
    assert recording() is None
