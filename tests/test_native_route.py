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


def test_out_proj_row_sums_are_formed_once(monkeypatch):
    """The kept row sums of out_proj's weight in another type: the weight is cast when they are formed, not
    at every forward, and they follow the weight's version and storage into the same buffer."""
    blk = HdcMamba9v3Block(64, 8, 2, 8)
    casts = []

    def row_sums(w, out=None):
        casts.append(w.dtype)
        s = w.detach().float().sum(1)
        return s if out is None else out.copy_(s)

    monkeypatch.setattr(_ops, "row_sums", row_sums)
    with torch.no_grad():
        a = blk._out_weight_sums(torch.bfloat16)
        assert blk._out_weight_sums(torch.bfloat16) is a and casts == [torch.bfloat16]
        blk.out_proj.weight.add_(1.0)
        before = a.clone()
        blk.refresh_derived_weights()
        blk.refresh_derived_weights()
        assert len(casts) == 2 and blk._out_weight_sums(torch.bfloat16) is a
        assert ((a - before) / 72 - 1).abs().max() < 0.01
