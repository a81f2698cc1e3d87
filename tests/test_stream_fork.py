"""A forked child does not take over the parent's way to the current stream: its
first call goes through torch.cuda.current_stream(), which refuses a process
whose GPU runtime was initialised before the fork."""
import os

from kvforge_amd import runtime as R


def test_child_asks_torch_again(monkeypatch):
    import torch
    calls = []
    monkeypatch.setattr(R, "_current_raw", lambda: calls.append(1) or 7)
    assert R.stream_handle().value == 7 and calls == [1]

    def refuse():
        raise RuntimeError("forked")

    monkeypatch.setattr(torch.cuda, "current_stream", refuse)
    pid = os.fork()
    if pid == 0:
        try:
            R.stream_handle()
        except RuntimeError as e:
            os._exit(0 if str(e) == "forked" else 2)
        os._exit(1)
    assert os.waitstatus_to_exitcode(os.waitpid(pid, 0)[1]) == 0
    assert R.stream_handle().value == 7  # the parent keeps its own
