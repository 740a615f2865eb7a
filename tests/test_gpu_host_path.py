"""The native call path against the Python path: same bits, same gradients, same
refusals, over the forms of calls that either may get; and what sits between a
call and the device (no_grad, saved-tensor hooks, checkpointing, functorch,
forward mode, tensor subclasses, modes, threads, streams)."""
import threading

import pytest
import torch
import torch.autograd.forward_ad as fwad
from torch.utils.checkpoint import checkpoint

import smooth_attn
from smooth_attn import _lib, kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"


class _NoNative:
    """Answers as the native path does to a call it does not take."""

    def __init__(self):
        self.asked = 0

    def _none(self, *a):
        self.asked += 1

    causal_norm = flash = paged = paged_append = _none

    def norm_out(self, *a):
        self.asked += 1
        return False


class _Counting:
    """The native path, counting the calls that it took."""

    def __init__(self):
        self.took = 0

    def __getattr__(self, name):
        fn = getattr(_lib.host(), name)

        def call(*a):
            r = fn(*a)
            self.took += r is not None and name != "norm_out"  # (the Python path asks for that one too)
            return r
        return call


def both(monkeypatch, call):
    """call() on the Python path and on the native one: (Python, native, times the native path took it)."""
    got = []
    for nat in (_NoNative(), _Counting()):
        monkeypatch.setattr(kernels, "_native", lambda nat=nat: nat)
        try:
            got.append(call())
        except Exception as e:  # noqa: BLE001
            got.append(e)
    monkeypatch.undo()
    return got[0], got[1], nat.took


def same(a, b):
    if isinstance(a, Exception) or isinstance(b, Exception):
        assert type(a) is type(b), (a, b)
        return
    if isinstance(a, torch.Tensor):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
        assert a.requires_grad == b.requires_grad and type(a) is type(b)
        a, b = (torch.empty(t.numel(), dtype=t.dtype, device=t.device).copy_(t.detach().reshape(-1)).view(torch.uint8)
                for t in (a, b))
        assert torch.equal(a, b)
        return
    assert len(a) == len(b)
    for x, y in zip(a, b):
        same(x, y)


def randn(*shape, dtype=torch.bfloat16, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _layouts(H, T, D, dtype, seed):
    """[2, H, T, D] tensors of one content type in the layouts a program may hold."""
    base = randn(2, H, T, D, dtype=dtype, seed=seed)
    yield "contiguous", base
    yield "bthd", randn(2, T, H, D, dtype=dtype, seed=seed).transpose(1, 2)
    yield "wide rows", randn(2, H, T, 2 * D, dtype=dtype, seed=seed)[..., D:]
    yield "off by one", randn(2 * H * T * D + 1, dtype=dtype, seed=seed)[1:].view(2, H, T, D)
    yield "d not last", randn(2, H, D, T, dtype=dtype, seed=seed).transpose(2, 3)
    yield "heads expanded", randn(2, 1, T, D, dtype=dtype, seed=seed).expand(2, H, T, D)
    yield "odd stride", randn(2, H, T, D + 1, dtype=dtype, seed=seed)[..., :D]
    yield "order", randn(T, 2, H, D, dtype=dtype, seed=seed).permute(1, 2, 0, 3)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("D", [8, 20, 64, 100])
def test_attention_layouts(monkeypatch, dtype, D):
    T, took = 70, 0
    for (n1, q), (n2, k) in zip(_layouts(4, T, D, dtype, 1), list(_layouts(2, T, D, dtype, 2))[::-1]):
        for qq, kk, vv in ((q, k, randn(2, 2, T, D, dtype=dtype, seed=3)), (randn(2, 4, T, D, dtype=dtype, seed=4), k, k)):
            for kw in ({}, {"window_size": 9}, {"scale": 0.3, "exact_math": True}):
                def call():
                    a = [t.detach().requires_grad_(True) for t in (qq, kk, vv)]
                    o = smooth_attn.sp2norm_flash_attention(*a, **kw)
                    do = randn(*o.shape, dtype=dtype, seed=5)
                    return [o, *torch.autograd.grad(o, a, do)]
                p, n, t = both(monkeypatch, call)
                same(p, n)
                took += t
                same(*both(monkeypatch, lambda: smooth_attn.sp2norm_flash_attention(qq, kk, vv, **kw))[:2])
    assert took > 0 or D % 8  # some of these forms are ordinary


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("L", [1, 33, 256])
def test_norm_forms(monkeypatch, dtype, L):
    fam = smooth_attn.FamilyConfig(alpha=1.5, theta=0.25, power=3)
    forms = [randn(2, 3, L, L, dtype=dtype), randn(L, L, dtype=dtype), randn(3, L, L, dtype=dtype).transpose(1, 2),
             randn(2, L, L + 1, dtype=dtype)[..., :L], randn(1, L, L, dtype=dtype).expand(2, L, L)]
    for x in forms:
        for kw in ({}, {"family": fam}, {"alpha": 3, "power": 1}):
            def train():
                a = x.detach().requires_grad_(True)
                y = smooth_attn.softplus_norm_causal(a, **kw)
                (dx,) = torch.autograd.grad(y, a, randn(*y.shape, dtype=dtype, seed=2))
                return [y, dx]
            p, n, took = both(monkeypatch, train)
            same(p, n)
            assert took == (1 if x.is_contiguous() else 0)
            for out in (torch.empty_like(x, memory_format=torch.contiguous_format),
                        torch.empty(*x.shape, 2, device=DEV, dtype=dtype)[..., 0]):
                p, n, _ = both(monkeypatch, lambda: smooth_attn.softplus_norm_causal_triton_out(out, x, **kw).clone())
                same(p, n)
            if x.dim() == 2:
                p, n, _ = both(monkeypatch, lambda: smooth_attn.softplus_norm_triton(x, **kw))
                same(p, n)


def test_refusals(monkeypatch):
    x = randn(2, 8, 8)
    q, k = randn(1, 4, 16, 64), randn(1, 2, 16, 64)
    calls = [
        lambda: smooth_attn.softplus_norm_causal(x[:, :4]),
        lambda: smooth_attn.softplus_norm_causal(x.int()),
        lambda: smooth_attn.softplus_norm_causal(x.cpu()),
        lambda: smooth_attn.softplus_norm_causal("x"),
        lambda: smooth_attn.softplus_norm_causal(randn(1, 1)[:0, :0]),
        lambda: smooth_attn.softplus_norm_causal_triton_out(x.float(), x),
        lambda: smooth_attn.softplus_norm_causal_triton_out(x[:1], x),
        lambda: smooth_attn.softplus_norm_triton_out(x, x),
        lambda: smooth_attn.softplus_norm_causal(x, family=smooth_attn.FamilyConfig(), alpha=1.0),
        lambda: smooth_attn.sp2norm_flash_attention(q, k.float(), k),
        lambda: smooth_attn.sp2norm_flash_attention(q, k, k[:, :1]),
        lambda: smooth_attn.sp2norm_flash_attention(q[:, :3], k, k),
        lambda: smooth_attn.sp2norm_flash_attention(q, k.cpu(), k),
        lambda: smooth_attn.sp2norm_flash_attention(q[0], k, k),
        lambda: smooth_attn.sp2norm_flash_attention(q, k, k, window_size=-1),
        lambda: smooth_attn.sp2norm_flash_attention(q, k, k, scale=float("nan")),
        lambda: smooth_attn.sp2norm_flash_attention(q[:, :, :0], k[:, :, :0], k[:, :, :0]),
    ]
    for c in calls:
        p, n, _ = both(monkeypatch, c)
        if isinstance(p, Exception):
            same(p, n)
            assert str(p) == str(n)
        else:
            assert torch.equal(torch.isnan(p), torch.isnan(n)) and torch.equal(p.nan_to_num(), n.nan_to_num())


@pytest.mark.parametrize("qd,cd", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                   (torch.float32, torch.float32), (torch.bfloat16, torch.float8_e4m3fn),
                                   (torch.float32, torch.bfloat16), (torch.float16, torch.float8_e4m3fn)])
@pytest.mark.parametrize("D", [24, 64, 128])
def test_paged_forms(monkeypatch, qd, cd, D):
    B, Hkv, P, W = 3, 2, 16, 5
    table = torch.randperm(B * W, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1)).view(B, W)
    lens = torch.tensor([70, 0, 33], device=DEV)
    caches = lambda: [randn(B * W, Hkv, P, D, seed=s).to(cd) for s in (2, 3)]
    forms = [caches(), [c.transpose(1, 2).contiguous().transpose(1, 2) for c in caches()]]
    if cd != torch.float8_e4m3fn:
        forms.append([torch.cat([c, c], -1)[..., :D] for c in caches()])
    # taken: one type for all (or bf16 q over e4m3fn caches), head dims of whole
    # 16-byte rows, int32 paging with unit strides
    pair = qd == cd or (qd, cd) == (torch.bfloat16, torch.float8_e4m3fn)
    row16 = 16 if cd == torch.float8_e4m3fn else 8
    for k, v in forms:
        for t, n in ((table.int(), lens.int()), (table, lens), (table.int().t().contiguous().t(), lens.int()),
                     (table.int(), torch.stack([lens.int(), lens.int()], 1)[:, 0])):
            paging = t.dtype == torch.int32 and t.stride(1) == 1 and n.dtype == torch.int32 and n.is_contiguous()
            q = randn(B, 4, 1, D, dtype=qd, seed=4)
            for qq in (q, randn(B, 1, 4, D, dtype=qd, seed=4).transpose(1, 2)):
                p, nat, took = both(monkeypatch, lambda: smooth_attn.sp2norm_paged_attention(qq, k, v, t, n))
                same(p, nat)
                assert took == (pair and paging and D % row16 == 0)
            for new in (randn(B, Hkv, 2, D, seed=5), randn(B, 2, Hkv, D, seed=5).transpose(1, 2)):
                def append():
                    kk, vv = k.clone(memory_format=torch.preserve_format), v.clone(memory_format=torch.preserve_format)
                    nn = new.to(cd)
                    return [smooth_attn.sp2norm_paged_kv_append(kk, vv, nn, nn, t, n), kk, vv]
                p, nat, took = both(monkeypatch, append)
                same(p, nat)
                assert took == (paging and D % row16 == 0)


def _train(x):
    y = smooth_attn.softplus_norm_causal(x)
    return torch.autograd.grad(y, x, torch.ones_like(y))[0]


def test_grad_modes_and_parameters(monkeypatch):
    q, k = randn(1, 4, 40, 64), randn(1, 2, 40, 64)
    for mode in (torch.no_grad, torch.inference_mode, torch.enable_grad):
        def call():
            with mode():
                a = torch.nn.Parameter(q.clone())
                o = smooth_attn.sp2norm_flash_attention(a, k, k)
                y = smooth_attn.softplus_norm_causal(torch.nn.Parameter(q[..., :40].contiguous()))
                return [o, y]
        p, n, took = both(monkeypatch, call)
        same(p, n)
        assert took == 2
    # only some inputs need gradients
    def some():
        kk = k.clone().requires_grad_(True)
        return torch.autograd.grad(smooth_attn.sp2norm_flash_attention(q, kk, k), kk, randn(1, 4, 40, 64, seed=3))
    same(*both(monkeypatch, some)[:2])


def test_saved_tensor_hooks_and_checkpoint(monkeypatch):
    q, k = randn(1, 4, 40, 64), randn(1, 2, 40, 64)

    def hooked():
        packed = []
        def pack(t):
            packed.append(tuple(t.shape))
            return t.cpu()
        a, x = q.clone().requires_grad_(True), q[..., :40].clone().requires_grad_(True)
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(DEV)):
            o = smooth_attn.sp2norm_flash_attention(a, k, k)
            y = smooth_attn.softplus_norm_causal(x)
        n = len(packed)
        g = torch.autograd.grad([o, y], [a, x], [torch.ones_like(o), torch.ones_like(y)])
        return [torch.tensor(n), *g]
    same(*both(monkeypatch, hooked)[:2])

    def checkpointed():
        a = q.clone().requires_grad_(True)
        o = checkpoint(lambda t: smooth_attn.sp2norm_flash_attention(t, k, k), a, use_reentrant=False)
        return torch.autograd.grad(o, a, torch.ones_like(o))
    same(*both(monkeypatch, checkpointed)[:2])

    def changed():  # a saved input changed in place is refused
        a = q.clone().requires_grad_(True)
        b = a * 1
        o = smooth_attn.sp2norm_flash_attention(b, k, k)
        b.add_(1)
        return torch.autograd.grad(o, a, torch.ones_like(o))
    p, n, _ = both(monkeypatch, changed)
    assert isinstance(p, RuntimeError) and isinstance(n, RuntimeError)


def _hooked(fn, unpack, *inputs):
    """Gradients of fn(*inputs) whose saved tensors came back through unpack."""
    a = [t.clone(memory_format=torch.preserve_format).requires_grad_(True) for t in inputs]
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach(), unpack):
        y = fn(*a)
    return torch.autograd.grad(y, a, randn(*y.shape, dtype=y.dtype, seed=9))


def _permuted(t):  # values as before, the last two dims swapped in memory
    return t.transpose(-1, -2).contiguous().transpose(-1, -2)


def _padded_rows(t):  # values as before, rows 3 elements apart
    return torch.cat([t, t[..., :3]], -1)[..., : t.shape[-1]]


def _off_by_one(t):
    return torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view(t.shape)


@pytest.mark.parametrize("unpack", [_permuted, _padded_rows, _off_by_one, lambda t: t.float(),
                                    lambda t: t.to(torch.float16)])
@pytest.mark.parametrize("shape", [(2, 3, 40, 40), (96, 96)])
def test_norm_backward_of_unpacked_forms(monkeypatch, unpack, shape):
    # a saved x of any layout or type of the kernels: the gradient of its values
    x = randn(*shape)
    p, n, took = both(monkeypatch, lambda: _hooked(smooth_attn.softplus_norm_causal, unpack, x))
    same(p, n)
    assert took == 1 and not isinstance(n, Exception)
    if unpack in (_permuted, _padded_rows, _off_by_one):
        # rows at another alignment sum in another order: fp32 noise, then at most one bf16 step
        (want,) = _hooked(smooth_attn.softplus_norm_causal, lambda t: t, x)
        assert torch.allclose(n[0].float(), want.float(), rtol=2.0 ** -7, atol=1e-5 * float(want.abs().max()))


@pytest.mark.parametrize("shape", [(3, 40, 40), (40, 40)])
def test_norm_backward_of_expanded_x(monkeypatch, shape):
    row = randn(1, 40)
    x = row.expand(shape).contiguous()
    p, n, _ = both(monkeypatch, lambda: _hooked(smooth_attn.softplus_norm_causal, lambda t: row.expand(shape), x))
    same(p, n)
    same(n, _hooked(smooth_attn.softplus_norm_causal, lambda t: t, x))


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.float16, 40), (torch.float32, 20)])
@pytest.mark.parametrize("unpack", [_permuted, _padded_rows, _off_by_one, lambda t: t.float()])
def test_attention_backward_of_unpacked_forms(monkeypatch, unpack, dtype, D):
    f = lambda q, k: smooth_attn.sp2norm_flash_attention(q, k, k, window_size=30)
    q, k = randn(2, 4, 70, D, dtype=dtype), randn(2, 2, 70, D, dtype=dtype, seed=1)
    fix = lambda t: unpack(t) if t.dim() == 4 else t  # (the row sums stay fp32 and dense)
    p, n, took = both(monkeypatch, lambda: _hooked(f, fix, q, k))
    same(p, n)
    assert took == 1 and not isinstance(n, Exception)
    if unpack in (_permuted, _padded_rows, _off_by_one):
        for a, b in zip(n, _hooked(f, lambda t: t, q, k)):
            assert torch.equal(a, b)


def test_attention_backward_of_a_type_with_fewer_head_dims(monkeypatch):
    # fp32 takes D = 20, the 16-bit types multiples of 8: padded, as the Python path does
    f = lambda q, k: smooth_attn.sp2norm_flash_attention(q, k, k)
    half = lambda t: t.to(torch.bfloat16) if t.dim() == 4 else t
    p, n, _ = both(monkeypatch, lambda: _hooked(f, half, randn(1, 4, 33, 20, dtype=torch.float32),
                                                randn(1, 2, 33, 20, dtype=torch.float32, seed=1)))
    assert not isinstance(n, Exception)
    same(p, n)


@pytest.mark.parametrize("which", ["q", "k", "o", "row sums", "all", "size"])
def test_attention_backward_refuses_mixed_saved_types(monkeypatch, which):
    # tensors that the kernels would read by another type's width or size
    f = lambda q, k: smooth_attn.sp2norm_flash_attention(q, k, k)
    q, k = randn(1, 4, 33, 64), randn(1, 2, 33, 64, seed=1)

    def call():
        seen = []

        def unpack(t):
            name = ["q", "k", "v", "o", "row sums"][len(seen)]
            seen.append(name)
            if which == "size":
                return t[:, :, :-1] if name == "k" else t
            return t.half() if which in (name, "all") else t
        return _hooked(f, unpack, q, k)
    for got in both(monkeypatch, call)[:2]:
        assert isinstance(got, ValueError), got


def test_norm_backward_refuses_saved_x_of_another_size():
    with pytest.raises(ValueError, match="grad_output's shape"):
        _hooked(smooth_attn.softplus_norm_causal, lambda t: t[:1], randn(2, 16, 16))


@pytest.mark.parametrize("entry", ["norm_out", "causal_norm", "causal_norm grad", "flash", "flash grad", "paged",
                                   "paged_append"])
def test_other_python_threads_run_during_a_launch(entry):
    # a launch that waits (a full queue, a first load of its code) must not stop
    # the interpreter.  In place of every launch the path calls PyGILState_Check,
    # whose 1 (this thread holds the interpreter) is an error status here.
    import ctypes

    addr = {n: ctypes.cast(getattr(_lib.load(), n), ctypes.c_void_p).value for n in _lib.SIGNATURES}
    check = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    launches = ("sa_norm_fwd", "sa_norm_bwd", "sa_flash_fwd", "sa_flash_bwd_ws", "sa_paged_decode",
                "sa_paged_kv_append_lens")
    x, q, k = randn(2, 32, 32), randn(1, 4, 40, 64), randn(1, 2, 40, 64)
    cache = torch.zeros(4, 2, 16, 64, device=DEV, dtype=torch.bfloat16)
    table = torch.zeros(1, 4, device=DEV, dtype=torch.int32)
    lens = torch.ones(1, device=DEV, dtype=torch.int32)
    host = _lib.host()
    host.bind({**addr, **{n: check for n in launches}})
    try:
        if entry == "norm_out":
            assert host.norm_out(torch.empty_like(x), x, True, 2.0, 0.5, 2)
        elif entry.startswith("causal_norm"):
            y = host.causal_norm(x.requires_grad_("grad" in entry), 2.0, 0.5, 2)
            if y.requires_grad:
                y.sum().backward()
        elif entry.startswith("flash"):
            o = host.flash(q.requires_grad_("grad" in entry), k, k, None, 0, False)
            if o.requires_grad:
                o.sum().backward()
        elif entry == "paged":
            assert host.paged(q[:, :, :1], cache, cache, table, lens, None, 16) is not None
        else:
            new = k[:, :, :1].contiguous()
            assert host.paged_append(cache, cache, new, new, table, lens, 16) is not None
    finally:
        host.bind(addr)


def test_errors_of_hooks_and_allocations_reach_the_caller():
    q, k = randn(1, 4, 40, 64), randn(1, 2, 40, 64)

    def pack(t):
        raise KeyError("from the hook")
    for fn in (lambda: smooth_attn.sp2norm_flash_attention(q.clone().requires_grad_(True), k, k),
               lambda: smooth_attn.softplus_norm_causal(q[..., :40].clone().requires_grad_(True))):
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t), pytest.raises(KeyError, match="from the hook"):
            fn()
    same(smooth_attn.sp2norm_flash_attention(q, k, k), smooth_attn.sp2norm_flash_attention(q.clone(), k, k))


def test_transforms_and_subclasses(monkeypatch):
    x = randn(3, 16, 16)
    q = randn(2, 2, 16, 32)

    class Sub(torch.Tensor):
        pass

    def dual():
        with fwad.dual_level():
            return smooth_attn.softplus_norm_causal(fwad.make_dual(x, torch.ones_like(x)))

    calls = [
        lambda: torch.func.vmap(smooth_attn.softplus_norm_causal)(x),
        lambda: torch.func.vmap(lambda t: smooth_attn.sp2norm_flash_attention(t[None], t[None], t[None]))(q),
        lambda: torch.func.grad(lambda t: smooth_attn.softplus_norm_causal(t).float().sum())(x),
        dual,
    ]
    for c in calls:
        p, n, took = both(monkeypatch, c)
        same(p, n)
        assert took == 0
    p, n, took = both(monkeypatch, lambda: smooth_attn.softplus_norm_causal(x.as_subclass(Sub)).as_subclass(torch.Tensor))
    same(p, n)
    assert took == 0
    with torch.device(DEV):  # a function mode
        p, n, took = both(monkeypatch, lambda: smooth_attn.softplus_norm_causal(x))
    same(p, n)
    assert took == 0

    def compiled():
        torch._dynamo.reset()
        return torch.compile(lambda t: smooth_attn.softplus_norm_causal(t * 1) + 1, backend="eager")(x)
    same(*both(monkeypatch, compiled)[:2])

    def double():
        a = x.clone().requires_grad_(True)
        y = smooth_attn.softplus_norm_causal(a)
        (g,) = torch.autograd.grad(y, a, torch.ones_like(y), create_graph=True)
        return [g]
    same(*both(monkeypatch, double)[:2])


def test_threads_and_streams():
    xs = [randn(4, 64, 64, seed=s).requires_grad_(True) for s in range(4)]
    want = [_train(x) for x in xs]
    got = [None] * 4

    def work(i):
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(s):
            for _ in range(20):
                got[i] = _train(xs[i])
        s.synchronize()
    torch.cuda.synchronize()
    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for a, b in zip(want, got):
        assert torch.equal(a, b)
