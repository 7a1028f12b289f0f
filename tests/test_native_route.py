"""Which calls take the native host path (no GPU: the rule alone)."""
import torch
from torch.autograd import forward_ad

from hdcmamba_amd import HdcMamba9v3Block, _ops


def test_native_path_rule(monkeypatch):
    """Everything but empty inputs, wide heads, other types, timed launches, unknown placements of the
    scan, autocast to another type and forward-mode differentiation (whose level torch keeps in a
    private name: it has to be there, for torch.func.jvp too)."""
    blk = HdcMamba9v3Block(64, 8, 2, 8)
    x = torch.zeros(1, 8, 64)
    assert blk._native_ok(x) and blk._native_ok(x.bfloat16())
    assert not blk._native_ok(x.half()) and not blk._native_ok(x[:0])
    assert not HdcMamba9v3Block(512, 8, 2, 8)._native_ok(x)
    with forward_ad.dual_level():
        assert not blk._native_ok(x)
    seen = []
    torch.func.jvp(lambda t: (t, seen.append(blk._native_ok(x)))[0], (x,), (x,))
    assert seen == [False] and blk._native_ok(x)
    with monkeypatch.context() as m:
        m.setattr(torch, "is_autocast_enabled", lambda device: device == "cuda")
        m.setattr(torch, "get_autocast_dtype", lambda device: torch.bfloat16)
        assert not blk._native_ok(x) and blk._native_ok(x.bfloat16())
    with monkeypatch.context() as m:
        m.setattr(_ops.timer, "active", {"ssm"})
        assert not blk._native_ok(x)
    blk.ssm_overlap = "unknown"
    assert not blk._native_ok(x)
