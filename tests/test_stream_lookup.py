"""The cached lookup of torch's current stream, on the CPU."""
import os

import pyc_amd


def test_forked_child_looks_the_stream_up_again(monkeypatch):
    """A child of a process that has used the device must go through
    torch.cuda.current_stream(), which refuses it, not through the parent's raw lookup."""
    monkeypatch.setattr(pyc_amd, "_current_raw_stream", lambda: 7)
    assert pyc_amd._stream(None) == 7
    pid = os.fork()
    if pid == 0:
        os._exit(0 if pyc_amd._current_raw_stream is None else 1)
    assert os.waitstatus_to_exitcode(os.waitpid(pid, 0)[1]) == 0
    assert pyc_amd._stream(None) == 7
