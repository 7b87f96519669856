"""The native calls of csrc/torch_calls.cpp against the general path of the Python modules, which
``_lib.calls`` switched off leaves in place: the same kernels on the same inputs, so the same bits, for
every form the native calls take; what they leave alone goes, and fails, the general way."""
import pytest
import torch
import torch.utils.checkpoint
from torch.autograd import forward_ad

from gpt_neox_amd import _lib, fused_rope
from gpt_neox_amd.fused_kernels import load, load_fused_kernels
from gpt_neox_amd.fused_softmax import FusedScaleMaskSoftmax, SoftmaxFusionTypes
from gpt_neox_amd.positional_embeddings import (AliBi, apply_rotary_pos_emb, apply_rotary_pos_emb_,
                                                apply_rotary_pos_emb_qkv_)

gpu = pytest.mark.gpu
DTYPES = [torch.float16, torch.bfloat16]


def module(dtype, fusion, scale=0.125):
    half = dtype == torch.float16
    return FusedScaleMaskSoftmax(half, not half, fusion, lambda x, m: x.masked_fill_(m, torch.finfo(x.dtype).min), True,
                                 scale, causal_mask_check="verify", skip_hidden_tails=False)


def both_ways(monkeypatch, fn):
    """``fn()`` through the native calls, which are counted, and without them."""
    served, real = [], _lib.load_calls()

    class Counting:
        def __getattr__(self, name):
            def call(*args, **kwargs):
                out = getattr(real, name)(*args, **kwargs)
                if out is not None and out is not False:
                    served.append(name)
                return out
            return call

    with monkeypatch.context() as m:
        m.setattr(_lib, "_calls", Counting())
        native = fn()
    with monkeypatch.context() as m:
        m.setattr(_lib, "calls", lambda *tensors: None)
        general = fn()
    return native, general, served


def causal_mask(s, device, window=None):
    hidden = torch.ones(s, s, dtype=torch.bool, device=device).triu_(1)
    if window is not None:
        hidden |= torch.ones(s, s, dtype=torch.bool, device=device).tril_(-window - 1)
    return hidden.view(1, 1, s, s)


SOFTMAX = [  # kind, b, np, sq, sk, call it is served by
    ("causal", 2, 3, 65, 65, "causal_softmax"),
    ("causal", 1, 1, 1, 1, "causal_softmax"),
    ("window", 1, 2, 648, 648, "causal_softmax"),
    ("alibi", 2, 4, 72, 72, "causal_softmax"),
    ("dropout", 2, 3, 96, 96, "causal_softmax"),
    ("alibi dropout", 2, 4, 40, 40, "causal_softmax"),
    ("masked", 3, 2, 33, 65, "masked_softmax"),
    ("masked batch", 3, 2, 64, 64, "masked_softmax"),
    ("decode", 4, 12, 1, 517, "masked_softmax"),
]


@gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("case", SOFTMAX, ids=lambda c: c[0])
def test_softmax_calls(device, monkeypatch, case, dtype):
    kind, b, np, sq, sk, served_by = case
    g = torch.Generator(device=device).manual_seed(3)
    x = (torch.randn(b, np, sq, sk, device=device, generator=g) * 8).to(dtype)
    dy = torch.randn(b, np, sq, sk, device=device, generator=g).to(dtype)
    if kind.startswith("masked") or kind == "decode":
        mb = b if kind == "masked batch" else 1
        mask = torch.rand(mb, 1, sq, sk, device=device, generator=g) < 0.4
        mod = module(dtype, SoftmaxFusionTypes.general)
    else:
        mask = causal_mask(sq, device, 100 if kind == "window" else None)
        mod = module(dtype, SoftmaxFusionTypes.upper_triang, 1)  # (an int scale, as the reference passes)
    kw = {}
    if "alibi" in kind:
        kw["alibi_slopes"] = AliBi(np, mp_size=1, mp_rank=0).slopes.to(device)
    if "dropout" in kind:
        kw["dropout_p"] = 0.25

    def run():
        torch.manual_seed(11)
        out = []
        if not kw.get("dropout_p"):
            with torch.no_grad():
                out.append(mod(x, mask, **kw))
        # (a contiguous gradient is overwritten)
        for grad in (dy.clone(), dy.clone().transpose(2, 3).contiguous().transpose(2, 3), dy[:, :, :1, :1].expand_as(dy)):
            xin = x.clone().requires_grad_(True)
            y = mod(xin, mask, **kw)
            out += [y.detach(), torch.autograd.grad(y, xin, grad)[0]]
        out.append(torch.tensor(torch.cuda.default_generators[0].get_offset()))
        return out

    native, general, served = both_ways(monkeypatch, run)
    assert all(torch.equal(a, c) for a, c in zip(native, general))
    assert served.count(served_by) == (3 if kw.get("dropout_p") else 4)


@gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("half_tables", [False, True])
@pytest.mark.parametrize("shape,heads_k,width,offset", [((7, 2, 3, 64), 3, 16, 0), ((1, 4, 12, 64), 12, 64, 20), ((5, 1, 8, 96), 2, 24, 3)])
def test_rotary_call(device, monkeypatch, shape, heads_k, width, offset, half_tables, dtype):
    s, b, h, hn = shape
    g = torch.Generator(device=device).manual_seed(5)
    mixed = torch.randn(s, b, h, 3 * hn, device=device, generator=g).to(dtype)
    angles = torch.randn(32, 1, 1, width, device=device, generator=g)
    cos, sin = angles.cos(), angles.sin()
    if half_tables:
        cos, sin = cos.to(dtype), sin.to(dtype)

    def run():
        q = mixed[..., :width].detach().requires_grad_(True)
        k = mixed[:, :, :heads_k, hn : hn + width].detach().requires_grad_(True)
        with torch.no_grad():
            out = list(apply_rotary_pos_emb(q, k, cos, sin, offset))
        oq, ok = apply_rotary_pos_emb(q, k, cos, sin, offset)
        out += [oq.detach(), ok.detach()]
        out += torch.autograd.grad((oq, ok), (q, k), (oq.detach().clone(), ok.detach().transpose(2, 3).contiguous().transpose(2, 3)),
                                   retain_graph=True)
        out += torch.autograd.grad(oq.float().sum(), (q, k))  # k's gradient comes as zeros, q's as an expanded scalar
        return out

    native, general, served = both_ways(monkeypatch, run)
    assert all(torch.equal(a, c) and a.stride() == c.stride() for a, c in zip(native, general))
    assert served == ["rotary"] * 2


@gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("d,d2,sliced", [(96, 24, False), (64, 64, False), (64, 16, True)])
def test_rope_calls(device, monkeypatch, d, d2, sliced, transpose, dtype):
    g = torch.Generator(device=device).manual_seed(6)
    base = torch.randn(9, 2, 3, 2 * d, device=device, generator=g).to(dtype)
    t0 = base[..., :d] if sliced else base[..., :d].contiguous()
    freqs = torch.randn(9, 1, 1, d2, device=device, generator=g)

    def run():
        out = []
        for fn, tables in ((fused_rope.fused_apply_rotary_pos_emb, (freqs,)),
                           (fused_rope.fused_apply_rotary_pos_emb_cached, (freqs.cos(), freqs.sin())),
                           (fused_rope.fused_apply_rotary_pos_emb_cached, (freqs.cos().to(dtype), freqs.sin().to(dtype)))):
            t = t0.detach().requires_grad_(True)
            y = fn(t, *tables, transpose)
            out += [y.detach(), torch.autograd.grad(y, t, y.detach().clone())[0], fn(t0, *tables, transpose)]
        return out

    native, general, served = both_ways(monkeypatch, run)
    assert all(torch.equal(a, c) and a.stride() == c.stride() for a, c in zip(native, general))
    assert served == ["rope"] * 6


@gpu
def test_saved_tensors_go_through_hooks_and_version_checks(device):
    x = torch.randn(1, 2, 40, 40, device=device).half().requires_grad_(True)
    mod, mask = module(torch.float16, SoftmaxFusionTypes.upper_triang), causal_mask(40, device)
    dy = torch.randn_like(x)
    want = torch.autograd.grad(mod(x, mask), x, dy.clone())[0]
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.cpu(), lambda t: t.to(device)):
        y = mod(x, mask)
    assert len(packed) == 1 and torch.equal(torch.autograd.grad(y, x, dy.clone())[0], want)
    y = mod(x, mask)
    y.detach().mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y, x, dy.clone())
    y = mod(x, mask)
    torch.autograd.grad(y, x, dy.clone())
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y, x, dy.clone())


@gpu
def test_exceptions_of_saved_tensor_hooks_and_activation_checkpointing(device):
    x = torch.randn(1, 2, 40, 40, device=device).half().requires_grad_(True)
    mod, mask = module(torch.float16, SoftmaxFusionTypes.upper_triang), causal_mask(40, device)
    q = torch.randn(4, 1, 2, 16, device=device).half().requires_grad_(True)
    cos, sin = torch.randn(2, 8, 1, 1, 16, device=device)
    freqs = torch.randn(4, 1, 1, 16, device=device)

    class Stop(Exception):
        pass

    def stop(t):
        raise Stop

    calls = (lambda: mod(x, mask), lambda: apply_rotary_pos_emb(q, q, cos, sin)[0],
             lambda: fused_rope.fused_apply_rotary_pos_emb(q, freqs))
    for call in calls:
        with pytest.raises(Stop), torch.autograd.graph.saved_tensors_hooks(stop, lambda t: t):
            call()
    # recomputed segments stop, by an exception from the pack hook, at the last tensor that is saved: in this call
    for leaf, call in zip((x, q, q), calls):
        want = torch.autograd.grad(call().float().pow(2).sum(), leaf)[0]
        y = torch.utils.checkpoint.checkpoint(lambda _: call(), leaf, use_reentrant=False)
        assert torch.equal(torch.autograd.grad(y.float().pow(2).sum(), leaf)[0], want)


@gpu
@pytest.mark.parametrize("native", [True, False])
def test_tables_that_a_saved_tensor_hook_gives_back(device, monkeypatch, native):
    # whatever the hook returns is checked on the host again before a kernel reads it
    if not native:
        monkeypatch.setattr(_lib, "calls", lambda *tensors: None)
    q = torch.randn(4, 1, 2, 16, device=device).half().requires_grad_(True)
    mixed = torch.randn(4, 1, 2, 48, device=device).half().requires_grad_(True)
    cos, sin = torch.randn(2, 6, 1, 1, 16, device=device)
    forward = [
        lambda: apply_rotary_pos_emb(q, q, cos, sin, 2)[0],
        lambda: apply_rotary_pos_emb_(q * 1, q * 1, cos, sin, 2)[0],
        lambda: apply_rotary_pos_emb_qkv_(mixed * 1, cos, sin, 2)[0],
        lambda: fused_rope.fused_apply_rotary_pos_emb(q, cos[:4]),
        lambda: fused_rope.fused_apply_rotary_pos_emb_cached(q, cos[:4], sin[:4]),
    ]

    def gradient(call, unpack):
        leaf = mixed if call is forward[2] else q
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: unpack(t) if t.dtype == torch.float32 else t):
            y = call()
        g = torch.ones_like(y)
        return torch.autograd.grad(y, leaf, g)[0]

    for call in forward:
        want = gradient(call, lambda t: t)
        # the same values in another layout
        assert torch.equal(gradient(call, lambda t: t.transpose(0, -1).contiguous().transpose(0, -1)), want)
        for unpack in (lambda t: t.cpu(), lambda t: t.double(), lambda t: t[:-1], lambda t: t.flatten()):
            with pytest.raises(RuntimeError):
                gradient(call, unpack)


@gpu
def test_forward_mode_derivatives_are_refused(device):
    # no kernel computes a tangent: an error, and not a result whose derivative has become zero
    t = torch.randn(4, 1, 2, 16, device=device).half()
    cos, sin = torch.randn(2, 4, 1, 1, 16, device=device)
    x = torch.randn(2, 4, 40, 40, device=device).half()
    wide = torch.randn(1, 2, 648, 648, device=device).half()
    causal, window = causal_mask(40, device), causal_mask(648, device, 100)
    some = torch.rand(1, 1, 40, 40, device=device) < 0.4
    padding = (torch.arange(40, device=device) >= 20).view(1, 1, 1, 40).expand(1, 1, 40, 40).contiguous()
    slopes = AliBi(4, mp_size=1, mp_rank=0).slopes.to(device)
    upper, general = (module(torch.float16, f) for f in (SoftmaxFusionTypes.upper_triang, SoftmaxFusionTypes.general))
    ends = FusedScaleMaskSoftmax(True, False, SoftmaxFusionTypes.general, None, True, 0.125, causal_mask_check="verify")
    calls = {  # name: (call, the arguments that may be dual)
        "rope": (fused_rope.fused_apply_rotary_pos_emb, (t, cos)),
        "rope cached": (fused_rope.fused_apply_rotary_pos_emb_cached, (t, cos, sin)),
        "rotary": (apply_rotary_pos_emb, (t, t.clone(), cos, sin)),
        "rotary in place": (apply_rotary_pos_emb_, (t.clone(), t.clone(), cos, sin)),
        "rotary of a projection": (apply_rotary_pos_emb_qkv_, (torch.randn(4, 1, 2, 48, device=device).half(), cos, sin)),
        "causal": (lambda x: upper(x, causal), (x,)),
        "window": (lambda x: upper(x, window), (wide,)),
        "mask": (lambda x: general(x, some), (x,)),
        "mask with row ends": (lambda x: ends(x, padding), (x,)),
        "alibi": (lambda x, s: upper(x, causal, alibi_slopes=s), (x, slopes)),
        "dropout": (lambda x: upper(x, causal, dropout_p=0.25), (x,)),
        "alibi dropout": (lambda x, s: upper(x, causal, alibi_slopes=s, dropout_p=0.25), (x, slopes)),
    }
    passed = []
    for name, (call, args) in calls.items():
        for i, a in enumerate(args):
            with forward_ad.dual_level():
                dual = [forward_ad.make_dual(b, torch.ones_like(b)) if j == i else b for j, b in enumerate(args)]
                for grad in (True, False):
                    try:
                        with torch.set_grad_enabled(grad):
                            call(*dual)
                        passed.append((name, i, grad))
                    except NotImplementedError as e:
                        assert "jvp" in str(e)
        call(*args)  # and outside of the level as ever
    assert not passed


@gpu
def test_native_calls_run_on_the_current_stream(device):
    x = torch.randn(2, 4, 200, 200, device=device).half()
    mod, mask, dy = module(torch.float16, SoftmaxFusionTypes.upper_triang), causal_mask(200, device), torch.randn_like(x)
    leaf = x.clone().requires_grad_(True)
    want = mod(leaf, mask)
    want_dx = torch.autograd.grad(want, leaf, dy.clone())[0]
    late, late_dy = torch.zeros_like(x).requires_grad_(True), torch.zeros_like(dy)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)  # the inputs arrive late, on this stream
        with torch.no_grad():
            late.copy_(x)
        y = mod(late, mask)
        torch.cuda._sleep(20_000_000)
        late_dy.copy_(dy)
        (dx,) = torch.autograd.grad(y, late, late_dy)
    side.synchronize()
    assert torch.equal(y, want) and torch.equal(dx, want_dx)


@gpu
def test_what_the_native_calls_leave_alone(device, monkeypatch):
    q = torch.randn(4, 1, 2, 16, device=device).half()
    cos, sin = torch.randn(2, 8, 1, 1, 16, device=device)
    freqs = torch.randn(4, 1, 1, 16, device=device)
    bad = [
        lambda: apply_rotary_pos_emb(q, q, cos[:3], sin[:3]),                 # too few positions
        lambda: apply_rotary_pos_emb(q, q, cos[..., :8], sin[..., :8]),       # another width
        lambda: apply_rotary_pos_emb(q, q, cos, sin, 5),
        lambda: fused_rope.fused_apply_rotary_pos_emb(q, freqs[:3]),
        lambda: fused_rope.fused_apply_rotary_pos_emb(q, freqs.half()),
        lambda: fused_rope.fused_apply_rotary_pos_emb(q.float(), freqs),
        lambda: fused_rope.fused_apply_rotary_pos_emb_cached(q, freqs, freqs.half()),
        lambda: module(torch.float16, SoftmaxFusionTypes.general)(q, torch.zeros(1, 1, 3, 3, dtype=torch.bool, device=device)),
        lambda: torch.func.vmap(lambda t: apply_rotary_pos_emb(t, t, cos, sin)[0])(q[None]),
    ]
    for call in bad:
        errors = []

        def run():
            with pytest.raises(Exception) as e:
                call()
            errors.append((type(e.value), str(e.value).split("\n")[0]))

        _, _, served = both_ways(monkeypatch, run)
        assert errors[0] == errors[1] and not served
    # other layouts are served the general way
    flipped = cos.flip(0).transpose(0, 3).contiguous().transpose(0, 3)
    native, general, served = both_ways(monkeypatch, lambda: apply_rotary_pos_emb(q, q, flipped, flipped))
    assert all(torch.equal(a, c) for a, c in zip(native, general)) and not served


def test_no_native_call_for_cpu_tensors_subclasses_or_traces():
    class Marked(torch.Tensor):
        pass

    t = torch.zeros(2, 2)
    assert _lib.calls(t) is None and _lib.calls(t.as_subclass(Marked)) is None
    seen = []

    def f(x):
        seen.append(_lib.calls(x))
        return x + 1

    torch.jit.trace(f, (t,), check_trace=False)
    assert seen == [None]
    assert _lib.load_calls() is _lib.load_calls()


def test_missing_native_calls_raise_import_error(monkeypatch):
    monkeypatch.setattr(_lib, "_calls", None)
    monkeypatch.setattr(_lib, "CALLS_PATH", "/nonexistent/neox_torch.so")
    with pytest.raises(ImportError, match="neox_torch.so"):
        _lib.load_calls()


@pytest.fixture
def without_native_calls(monkeypatch):
    """A tree in which only libneox_fused.so was built."""
    monkeypatch.setattr(_lib, "_calls", None)
    monkeypatch.setattr(_lib, "_calls_missing", False)
    monkeypatch.setattr(_lib, "CALLS_PATH", "/nonexistent/neox_torch.so")


def test_the_library_alone_is_enough_to_load(without_native_calls, monkeypatch):
    with pytest.warns(RuntimeWarning, match="neox_torch.so"):
        load_fused_kernels()
    load_fused_kernels()  # (said once)
    built = []
    monkeypatch.setattr(_lib, "build", lambda *args, **kwargs: built.append(args))
    load()
    assert _lib.find_calls() is None and not built


@gpu
def test_the_library_alone_serves_every_call(device, without_native_calls):
    x = torch.randn(2, 2, 40, 40, device=device).half().requires_grad_(True)
    with pytest.warns(RuntimeWarning, match="neox_torch.so"):
        mod = module(torch.float16, SoftmaxFusionTypes.upper_triang)
    mask = causal_mask(40, device)
    y = mod(x, mask)
    assert type(y.grad_fn).__name__ == "_CausalSoftmax4DBackward"
    want = torch.softmax((x.detach().float() * 0.125).masked_fill(mask, float("-inf")), -1)
    assert (y.float() - want).abs().max() <= 1e-3
    q, freqs = torch.randn(4, 1, 2, 16, device=device).half(), torch.randn(4, 1, 1, 16, device=device)
    assert torch.equal(apply_rotary_pos_emb(q, q, freqs.cos(), freqs.sin())[1],
                       fused_rope.fused_apply_rotary_pos_emb_cached(q, freqs.cos(), freqs.sin()))


@pytest.mark.parametrize("attr,value", [("abi_version", 3), ("torch_version", "1.0.0")])
def test_native_calls_of_another_build_are_not_used(monkeypatch, attr, value):
    real = _lib.importlib.util.module_from_spec

    def other(spec):
        module = real(spec)
        exec_module = spec.loader.exec_module
        monkeypatch.setattr(spec.loader, "exec_module", lambda m: (exec_module(m), setattr(m, attr, value)), raising=False)
        return module

    monkeypatch.setattr(_lib, "_calls", None)
    monkeypatch.setattr(_lib.importlib.util, "module_from_spec", other)
    with pytest.raises(ImportError, match="build it again"):
        _lib.load_calls()
