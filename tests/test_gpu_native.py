"""What the native host path owes its callers beyond equal values: every test runs on it and on the
Python composition of the same kernels, which states what is right, refused or accepted."""
import weakref

import pytest
import torch

from cfgs import max_rel, reinit_block_

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


def _block(dev, dtype=torch.float32, mixer=False, dm=256, ds=64, H=4, C=64, seed=3):
    from hdcmamba_amd import HdcMamba9v3Block

    torch.manual_seed(0)
    blk = reinit_block_(HdcMamba9v3Block(dm, ds, H, C, differentiable_mixer=mixer), seed=seed, decays_uniform=True)
    return blk.to(dtype).to(dev).train()


def _x(dev, L, dtype=torch.float32, B=2, dm=256, seed=5):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randn(B, L, dm, generator=g, device=dev).to(dtype)


def _paths(blk):
    """blk on the native host path, then on the composition."""
    yield "native"
    blk._native_ok = lambda x: False
    yield "composition"
    del blk._native_ok


LIM = {torch.float32: 1e-5, torch.bfloat16: 1.5e-2}  # as test_native_training_is_the_composition


@pytest.mark.parametrize("mixer", [False, True])
@pytest.mark.parametrize("how", ["data", "pointer"])
def test_training_reads_the_weight_of_the_call(dev, mixer, how):
    """A training forward uses out_proj's weight as it is at the call, whatever changed it: a write
    through ``.data`` or into the storage leaves the version counter alone.  The rows of `combined`
    have a mean of about 1 (GroupNorm's bias) and the weight's rows a sum, so stale row sums would
    show."""
    _say("training weight", mixer, how)
    blk = _block(dev, torch.bfloat16, mixer)
    with torch.no_grad():
        blk.group_norm.bias.add_(2.0)
        blk.in_proj.bias[3 * 64 + 3 * 256:] += 3.0
        blk.out_proj.weight.add_(0.02)
    w0 = blk.out_proj.weight.detach().clone()
    x = _x(dev, 100, torch.bfloat16)
    out = {}
    for path in _paths(blk):
        with torch.no_grad():
            blk.out_proj.weight.copy_(w0)
        blk(x)
        w = blk.out_proj.weight
        if how == "data":
            w.data.mul_(-1.5)
        else:
            torch.empty(0, dtype=w.dtype, device=dev).set_(w.untyped_storage(), 0, w.shape).mul_(-1.5)
        out[path] = blk(x)[0].detach()
    assert max_rel(out["native"], out["composition"]) <= LIM[torch.bfloat16]


def test_training_out_proj_is_the_composition(dev):
    """The training forward normalises `combined` in a pass of its own (two-pass variance) before
    out_proj, also where nothing requires a gradient: bit-identical to the composition."""
    _say("training out_proj")
    blk = _block(dev, torch.bfloat16)
    x = _x(dev, 128, torch.bfloat16)
    out = {}
    for path in _paths(blk):
        blk.requires_grad_(True)
        a = blk(x)[0].detach()
        blk.requires_grad_(False)
        out[path] = a, blk(x)[0]
    assert torch.equal(out["native"][0], out["composition"][0])
    assert torch.equal(out["native"][1], out["composition"][1])


@pytest.mark.parametrize("mixer", [False, True])
def test_training_input_changed_in_place(dev, mixer):
    """x changed between forward and backward: refused where the forward kept x itself, and without
    effect where it kept a copy of its own (padded or not contiguous)."""
    _say("training input in place", mixer)
    blk = _block(dev, mixer=mixer)
    grads = {}
    for path in _paths(blk):
        x = _x(dev, 128)
        y = blk(x)[0].sum()
        x.add_(1.0)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.backward()
        for L, view in ((100, lambda t: t), (128, lambda t: t.transpose(0, 1).contiguous().transpose(0, 1))):
            for change in (False, True):
                x = view(_x(dev, L))
                y = blk(x)[0].square().sum()
                if change:
                    x.add_(1.0)
                (grads[path, L, change],) = torch.autograd.grad(y, [blk.out_proj.weight])
    for (path, L, _), g in grads.items():
        assert max_rel(g, grads["composition", L, False]) <= 1e-4, (path, L)


@pytest.mark.parametrize("mixer,L", [(False, 128), (True, 128), (True, 100)])
def test_training_input_is_freed_and_hooked(dev, mixer, L):
    """The kept input goes through saved-tensor hooks, and is given back when the backward has run,
    not with the graph."""
    _say("training input kept", mixer, L)
    blk = _block(dev, mixer=mixer)
    for path in _paths(blk):
        seen = []

        def pack(t):
            seen.append(tuple(t.shape))
            return t.cpu()

        leaf = _x(dev, L).requires_grad_()
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(dev)):
            h = leaf * 1.0
            y = blk(h)[0].sum()
        assert (2, 128, 256) in seen, path
        a = torch.autograd.grad(y, [leaf, blk.out_proj.weight])
        h = leaf * 1.0
        y = blk(h)[0].sum()
        alive = weakref.ref(h)
        del h
        b = torch.autograd.grad(y, [leaf, blk.out_proj.weight])
        assert alive() is None, path
        assert all(max_rel(s, t) <= 1e-5 for s, t in zip(a, b)), path


@pytest.mark.parametrize("mixer,L", [(False, 128), (False, 100), (True, 128), (True, 100)])
def test_training_backward_with_frozen_parameters(dev, mixer, L):
    """With x alone requiring a gradient: the differentiable mixer keeps x, so a second backward through
    the freed graph raises; without it the gradient is dy itself, nothing is kept, and a second
    backward and a changed x are accepted."""
    _say("frozen parameters", mixer, L)
    blk = _block(dev, mixer=mixer).requires_grad_(False)
    grads = []
    for path in _paths(blk):
        x = _x(dev, L).requires_grad_()
        h = x + 0.0  # (keeps nothing itself)
        y = blk(h)[0].square().sum()
        grads.append(torch.autograd.grad(y, [x], retain_graph=True)[0])
        if mixer:
            torch.autograd.grad(y, [x])
            with pytest.raises(RuntimeError, match="second time"):
                torch.autograd.grad(y, [x])
        else:
            z = blk(h)[0].sum()
            h.add_(1.0)
            for _ in range(2):
                assert torch.equal(torch.autograd.grad(z, [x])[0], torch.ones_like(x)), path
    assert max_rel(*grads) <= 1e-5


@pytest.mark.parametrize("L", [128, 100])
def test_training_output_changed_in_place(dev, L):
    """The training output may be changed in place (a residual added to it), padded or not."""
    _say("training output in place", L)
    blk = _block(dev, mixer=True)
    grads = []
    for path in _paths(blk):
        x = _x(dev, L).requires_grad_()
        y, _ = blk(x)
        y += x
        y *= 2.0
        grads.append(torch.autograd.grad(y, [x, blk.out_proj.weight, blk.in_proj.weight], torch.ones_like(y)))
    assert all(max_rel(a, b) <= 1e-5 for a, b in zip(*grads))


@pytest.mark.parametrize("L", [128, 100])
def test_training_second_derivative(dev, L):
    """A gradient of a gradient with respect to x goes on to what x was made from, padded or not."""
    _say("second derivative", L)
    blk = _block(dev)
    res = []
    for path in _paths(blk):
        s = torch.ones((), device=dev, requires_grad=True)
        x = _x(dev, L)
        y, _ = blk(x * s)
        (gs,) = torch.autograd.grad((y ** 3).sum(), [s], create_graph=True)
        res.append(torch.stack([gs.detach(), torch.autograd.grad(gs, [s])[0]]))
    assert torch.isfinite(res[0]).all()
    assert ((res[0] - res[1]).abs() <= 1e-4 * res[1].abs()).all()


def test_training_gradients_in_the_parameters_types(dev):
    """Parameters kept in fp32 beside bf16 ones get gradients of fp32 sums that were not rounded to bf16 on
    the way (A_log and the GroupNorm's among the mixer's)."""
    _say("mixed parameter types")
    grads = []
    blk = _block(dev, torch.bfloat16, mixer=True)
    blk.A_log.data = blk.A_log.data.float()
    blk.group_norm.bias.data = blk.group_norm.bias.data.float()
    x = _x(dev, 128, torch.bfloat16)
    dy = _x(dev, 128, torch.bfloat16, seed=6)
    want = [blk.A_log, blk.group_norm.bias, blk.group_norm.weight]
    g = torch.autograd.grad(blk(x)[0], want, dy)
    assert [t.dtype for t in g] == [torch.float32, torch.float32, torch.bfloat16]
    for t in g[:2]:
        assert not torch.equal(t, t.bfloat16().float())
    grads.append(g)
    f = _block(dev, torch.float32, mixer=True)
    f.load_state_dict(blk.state_dict())
    f.norm.weight.data = f.norm.weight.data.bfloat16()  # the first of the LayerNorm + conv's
    h = torch.autograd.grad(f(x.float())[0], [f.norm.weight, f.norm.bias, f.conv1d.weight, f.conv1d.bias], dy.float())
    assert [t.dtype for t in h] == [torch.bfloat16] + 3 * [torch.float32]
    for t in h[1:]:
        assert not torch.equal(t, t.bfloat16().float())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C", [64, 50])  # without and with padding at 100 rows
def test_single_sequence_of_any_batch_stride(dev, dtype, C):
    """A batch of one may come with any batch stride (one sequence of a batch whose sequences are a few
    values apart), a token row likewise."""
    _say("batch stride", dtype, C)
    blk = _block(dev, dtype, C=C).eval()
    buf = torch.randn(2, 100 * 256 + 3, device=dev).to(dtype)
    x = buf[:, :100 * 256].view(2, 100, 256)[:1]
    xc = x.clone(memory_format=torch.contiguous_format)
    assert x.stride(0) % 4 == 3
    with torch.no_grad():
        assert torch.equal(blk(x)[0], blk(xc)[0])
        a, b = blk.prefill(x), blk.prefill(xc)
        assert torch.equal(a[0], b[0])
        assert torch.equal(blk.step(buf[:1, :256], a[1]), blk.step(buf[:1, :256].clone(memory_format=torch.contiguous_format), b[1]))
    blk.train()
    g = [torch.autograd.grad(blk(t)[0].sum(), [blk.out_proj.weight])[0] for t in (x, xc)]
    assert torch.equal(*g)


@pytest.mark.parametrize("H,dm", [(4, 192), (4, 256)])
def test_mixer_gradient_of_an_unaligned_upstream(dev, H, dm):
    """The mixer's upstream gradient may be contiguous at any address."""
    from hdcmamba_amd.model import SlotSsmMixerFunction

    _say("unaligned upstream gradient", H, dm)
    ds = 32
    projs = (0.5 * torch.randn(1, 64, 3 * ds + 4 * dm, device=dev)).requires_grad_()
    A = torch.log(torch.linspace(0.5, 2.0, ds, device=dev))
    out = SlotSsmMixerFunction.apply(projs, A, torch.full((H,), 0.95, device=dev), torch.ones(dm, device=dev),
                                     torch.zeros(dm, device=dev), ds, dm, H, 64)
    flat = torch.randn(out.numel() + 1, device=dev)
    dy = flat[1:].view(out.shape)
    a, b = (torch.autograd.grad(out, [projs], t, retain_graph=True)[0] for t in (dy, dy.clone()))
    assert torch.equal(a, b)


@pytest.mark.parametrize("mixer", [False, True])
@pytest.mark.parametrize("dtype,region", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float16)])
def test_training_backward_in_an_autocast_region(dev, mixer, dtype, region):
    """A backward called inside an autocast region that the forward was not in computes in the
    forward's types: the same gradients as outside."""
    _say("backward under autocast", mixer, dtype, region)
    blk = _block(dev, dtype, mixer)
    x = _x(dev, 100, dtype).requires_grad_()
    dy = _x(dev, 100, dtype, seed=6)
    params = [x, blk.out_proj.weight] + ([blk.in_proj.weight, blk.norm.weight, blk.A_log] if mixer else [])
    want = torch.autograd.grad(blk(x)[0], params, dy)
    y = blk(x)[0]
    with torch.amp.autocast("cuda", dtype=region):
        got = torch.autograd.grad(y, params, dy)
    assert all(a.dtype == b.dtype and torch.equal(a, b) for a, b in zip(got, want))


def test_step_refuses_a_state_elsewhere(dev):
    """A decode state left on the CPU, wholly or one tensor of it, is an error before any launch."""
    _say("step state device")
    blk = _block(dev, torch.bfloat16).eval()
    x = _x(dev, 64, torch.bfloat16)
    with torch.no_grad():
        _, st = blk.prefill(x)
        for path in _paths(blk):
            for name in ("conv", "h", "S_prev", "S_intra"):
                kept = getattr(st, name)
                setattr(st, name, kept.cpu())
                with pytest.raises(RuntimeError, match="cpu"):
                    blk.step(x[:, 0], st)
                setattr(st, name, kept)
            assert torch.isfinite(blk.step(x[:, 0], st)).all(), path
        with pytest.raises(RuntimeError, match="cpu"):
            blk.step(x[:, 0], st, pos_dev=torch.zeros(1, dtype=torch.int32))


def test_scan_overlap_from_threads_and_in_a_graph(dev):
    """The scan on the side stream gives the same rows from short-lived threads and from every replay of a
    recorded forward, with eager forwards between the replays."""
    import threading

    _say("overlap threads, graph")
    blk = _block(dev, torch.bfloat16).eval()
    x = _x(dev, 128, torch.bfloat16)
    with torch.no_grad():
        want = blk(x)[0]
        other = blk(-x)[0]
    for mode in ("none", "state", "gate", "after_state"):
        blk.ssm_overlap = mode
        got = []

        def work():
            with torch.no_grad():
                got.append(blk(x)[0])

        for _ in range(3):
            t = threading.Thread(target=work)
            t.start()
            t.join()
        assert len(got) == 3 and all(torch.equal(g, want) for g in got), mode
        xs = x.clone()
        with torch.no_grad():
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                y = blk(xs)[0]
            for k in range(4):
                xs.copy_(x if k % 2 else -x)
                graph.replay()
                assert torch.equal(blk(x)[0], want), (mode, k)
                torch.cuda.synchronize()
                assert torch.equal(y, want if k % 2 else other), (mode, k)


def test_training_on_two_streams(dev):
    """Two blocks trained from two threads, each on a stream of its own, get the gradients of one after the
    other: nothing but the weights' own storage is shared."""
    import threading

    _say("two streams")
    blocks = [_block(dev, torch.bfloat16, mixer=True, seed=s) for s in (3, 4)]
    xs = [_x(dev, L, torch.bfloat16, seed=L) for L in (1000, 700)]

    def step(i):
        blk, x = blocks[i], xs[i]
        y = blk(x)[0]
        return torch.autograd.grad(y, [blk.out_proj.weight, blk.in_proj.weight, blk.A_log], torch.ones_like(y))

    want = [step(i) for i in range(2)]
    torch.cuda.synchronize()
    got, errors = [[], []], []
    gate = threading.Barrier(2, timeout=60)

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream(dev)):
                step(i)
                gate.wait()
                got[i] = [step(i) for _ in range(8)]
                torch.cuda.current_stream(dev).synchronize()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for i in range(2):
        for g in got[i]:
            assert all(torch.equal(a, b) for a, b in zip(g, want[i])), i


def test_parameters_of_another_shape_are_refused(dev):
    """A projection that does not fit x, or a parameter that is too short, is an error before any launch."""
    _say("parameter shapes")
    blk = _block(dev, mixer=True)
    x = _x(dev, 64)
    ds, dm, N = 64, 256, 3 * 64 + 4 * 256
    swaps = [("in_proj", torch.nn.Linear(dm + 8, N)), ("in_proj", torch.nn.Linear(dm - 8, N)),
             ("out_proj", torch.nn.Linear(dm, dm, bias=False)), ("out_proj", torch.nn.Linear(ds + dm, dm - 8, bias=False)),
             ("group_norm", torch.nn.GroupNorm(4, dm - 64)), ("norm", torch.nn.LayerNorm(dm - 64))]
    for name, layer in swaps:
        kept = getattr(blk, name)
        setattr(blk, name, layer.to(dev))
        with pytest.raises(RuntimeError):
            blk(x)
        with torch.no_grad(), pytest.raises(RuntimeError):
            blk(x)
        with torch.no_grad(), pytest.raises(RuntimeError):
            blk.step(x[:, 0], blk.new_state(2, dev, x.dtype))
        setattr(blk, name, kept)
    blk.A_log.data = blk.A_log.data[:-1]
    with torch.no_grad(), pytest.raises(RuntimeError):
        blk(x)
    with torch.no_grad(), pytest.raises(RuntimeError):
        blk.step(x, blk.new_state(2, dev, x.dtype))  # (a token row has two dimensions)
