"""The Python binding in a forked child: the stream is asked of torch again, which refuses a device
that the parent initialised, as it did before the binding kept torch's raw getters."""
import os

import tcrv_hip


def in_child(check):
    """Exit status of a forked child that runs check()."""
    pid = os.fork()
    if pid == 0:
        status = 1
        try:
            status = 0 if check() else 2
        finally:
            os._exit(status)
    return os.waitstatus_to_exitcode(os.waitpid(pid, 0)[1])


def test_a_child_asks_torch_for_the_stream_again(monkeypatch):
    asked = []
    monkeypatch.setattr(tcrv_hip, "_raw_stream", lambda: 7)  # as after a call in the parent
    monkeypatch.setattr(tcrv_hip, "_raw_stream_getter", lambda: asked.append(1) or (lambda: 9))
    assert tcrv_hip._stream(None) == 7 and not asked
    assert in_child(lambda: tcrv_hip._stream(None) == 9 and asked == [1]) == 0
    assert tcrv_hip._stream(None) == 7
