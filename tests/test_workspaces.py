"""Rules of the workspaces that outlive a call, on the host alone (no GPU: the streams are stand-ins)."""
import contextlib

import pytest
import torch

from hdcmamba_amd import _ops


class _Stream:
    device = torch.device("cuda", 0)

    def __init__(self, handle):
        self.cuda_stream, self.after = handle, []

    def wait_stream(self, other):
        self.after.append(other)


@pytest.fixture
def streams(monkeypatch):
    """A main and a side stream; ``capturing`` holds the streams that are being recorded."""
    main, side, capturing = _Stream(1), _Stream(2), set()
    now = [main]

    @contextlib.contextmanager
    def on(s):
        now.append(s)
        yield
        now.pop()

    class Lib:
        hdcm_ssm_workspace_bytes = staticmethod(lambda B, L, ds: 1024 * B)

    class Native:
        MAIN, OVERLAP = 0, {"state": 2}

    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: now[-1])
    monkeypatch.setattr(torch.cuda, "stream", on)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: now[-1] in capturing)
    monkeypatch.setattr(_ops, "side_stream", lambda device: side)
    monkeypatch.setattr(_ops, "lib", lambda: Lib)
    monkeypatch.setattr(_ops, "native", lambda: Native)
    monkeypatch.setattr(_ops, "_ssm_ws", {})
    monkeypatch.setattr(_ops, "_ssm_ws_kept", [])
    return main, side, capturing


@pytest.mark.parametrize("overlap", ["auto", "state"])
def test_scan_workspace_is_not_made_in_a_capture(streams, overlap):
    """A capture without the workspace, or with too small a one, is refused: the buffer would be filled
    on the side stream, which is not recorded, with nothing to order the replays after it."""
    main, side, capturing = streams
    t = torch.empty(1, 4, 8)
    capturing.add(main)
    with pytest.raises(RuntimeError, match="before graph capture"):
        _ops.native_streams(t, 4, 64, overlap)
    capturing.clear()
    _ops.native_streams(t, 4, 64, overlap)
    capturing.add(main)
    with pytest.raises(RuntimeError, match="before graph capture"):
        _ops.native_streams(torch.empty(9, 4, 8), 4, 64, overlap)
    assert _ops.native_streams(t, 4, 64, overlap)[3] is _ops._ssm_ws[(0, 2)]  # the side stream's


def test_scan_workspace_fill_is_ordered_before_the_caller(streams):
    """The stream whose call makes the side stream's workspace waits for its zero fill, once."""
    main, side, _ = streams
    for _ in range(2):
        _ops.native_streams(torch.empty(1, 4, 8), 4, 64, "auto")
        assert main.after == [side]
