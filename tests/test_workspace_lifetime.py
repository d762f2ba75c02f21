"""How long a stream's launch scratch lives (no GPU: the HIP runtime is the fake of test_runtime_host)."""

from types import SimpleNamespace

import pytest

from krn_amd.runtime import hip, hipapi
from tests.test_runtime_host import fake  # noqa: F401


class Memory:
    """A device whose buffers are counted while something refers to them."""

    def __init__(self):
        self.live, self.most, self.log = 0, 0, []

    def empty_on(self, stream, dtype, nbytes):
        memory = self

        class Buffer:
            def __init__(self):
                self.nbytes, self.pointer = nbytes, 16
                memory.live += 1
                memory.most = max(memory.most, memory.live)
                memory.log.append("made")

            def __del__(self):
                memory.live -= 1
                memory.log.append("freed")

        return Buffer()


def launches(memory, nbytes):
    launch = hip.Launch(SimpleNamespace(name="split"), None)
    return launch._with_workspace(lambda workspace, stream: memory.log.append("launched"), nbytes)


def test_a_replay_loop_holds_one_buffer_above_what_a_stream_keeps(fake):  # noqa: F811
    """Stream-ordered memory is returned right after the launch that uses it (the free waits for that work), so replays
    never hold more than one, however far the device lags behind: no marker completes here."""
    memory = Memory()
    stream = hip.HIPStream(memory, 1)
    run = launches(memory, hip.WORKSPACE_KEPT + 1)
    for _ in range(600):
        run(stream)
    assert memory.most == 1 and memory.live == 0
    assert memory.log == ["made", "launched", "freed"] * 600


def test_a_failed_launch_returns_its_buffer(fake):  # noqa: F811
    memory = Memory()
    stream = hip.HIPStream(memory, 1)

    def call(workspace, handle):
        raise RuntimeError("refused")

    run = hip.Launch(SimpleNamespace(name="split"), None)._with_workspace(call, hip.WORKSPACE_KEPT + 1)
    with pytest.raises(RuntimeError, match="refused"):
        run(stream)
    assert memory.live == 0 and not stream.workspace_lock.locked()


def test_smaller_requests_share_one_buffer_that_grows(fake):  # noqa: F811
    memory = Memory()
    stream = hip.HIPStream(memory, 1)
    small, large = launches(memory, 64), launches(memory, 128)
    for run in (small, small, large, small, large):
        run(stream)
    assert memory.log == ["made", "launched", "launched", "made", "freed", "launched", "launched", "launched"]


def test_a_graph_keeps_the_buffers_of_the_launches_it_records(fake, monkeypatch):  # noqa: F811
    memory = Memory()
    stream = hip.HIPStream(memory, 1)
    monkeypatch.setattr(hipapi, "capturing", lambda handle: True)
    for nbytes in (64, hip.WORKSPACE_KEPT + 1):
        launches(memory, nbytes)(stream)
    held = stream.take()
    assert memory.live == 2 and len(held) == 2
    del held
    assert memory.live == 0
