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


def test_product_rules_at_their_lines():
    """Which products run on the kernels here: both sides of every line of the rules."""
    lib = _ops.lib()
    f32 = lib.hdcm_gemm_f32_preferred
    assert f32(64, 4480, 1024) and f32(8192, 4480, 1024) and f32(1000, 1024, 1152) and not f32(63, 4480, 1024)
    assert not f32(16384, 4480, 1024) and not f32(512, 1408, 1472) and not f32(256, 6336, 1536)
    tn = lambda M, N, K, sums: lib.hdcm_gemm_tn_preferred(M, N, K, sums, _ops.HDCM_BF16)  # noqa: E731
    assert tn(1024, 2240, 512, 1) and not tn(1023, 2240, 512, 1) and tn(4096, 768, 832, 0) and not tn(4095, 768, 832, 0)
    for N, K in ((6336, 1536), (8576, 2048)):  # one partial round of split tiles more than the library
        assert tn(4095, N, K, 1) and not tn(4096, N, K, 1) and not tn(10240, N, K, 1) and tn(10241, N, K, 1)
    assert tn(8192, 5184, 1280, 1) and tn(8192, 10624, 2560, 1)
    bf = lambda M, N, K: lib.hdcm_gemm_preferred(M, N, K, _ops.HDCM_BF16)  # noqa: E731
    assert bf(32768, 3264, 768) and not bf(32769, 3264, 768) and bf(16384, 4480, 1024) and not bf(16385, 4480, 1024)
    assert not bf(8192, 6336, 1536) and not bf(0, 3264, 768) and not lib.hdcm_gemm_preferred(8192, 3264, 768, 0)
