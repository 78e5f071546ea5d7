"""The native loops of the Python face: which tensors they take and which they leave to the Python code (CPU), and that
both ways give the same bits (GPU)."""
import ctypes as C

import pytest
import torch
from torch.overrides import BaseTorchFunctionMode

from eridiffusion_amd import _lib as L
from eridiffusion_amd import _torch_face


class Sub(torch.Tensor):
    pass


def _handles(params):
    arr = (C.c_void_p * len(params))()
    for i, p in enumerate(params):
        h = C.c_void_p()
        tag = L.DTYPE_BF16 if p.dtype == torch.bfloat16 else L.DTYPE_F32
        L.check(L.lib().eri_param_create(p.data_ptr() or 1, p.numel(), tag, C.byref(h)), "eri_param_create")
        arr[i] = h
    return arr


def _gradient_forms(device):
    """(parameter, gradient, taken natively) of every form the list optimizer accepts."""
    bf, f32 = torch.bfloat16, torch.float32

    def new(*shape, dtype=f32, seed=11):
        return (torch.randn(*shape, generator=torch.Generator().manual_seed(sum(shape) + seed)) * 1e-3).to(dtype).to(device)
    leaf = new(40, 64).requires_grad_()
    param = torch.nn.Parameter(new(2049))
    return [(new(40, 64), new(40, 64), True), (new(40, 64, dtype=bf), new(40, 64, dtype=bf), True),
            (new(40, 64, dtype=bf), new(40, 64), True),              # fp32 gradient of a bf16 parameter
            (new(40, 64), new(40, 64, dtype=bf), False),             # cast to the parameter's dtype
            (new(40, 64), new(64, 40).t(), False),                   # transposed
            (new(64), new(64, 2)[:, 0], False),                      # strided
            (new(40, 64), new(40, 64).as_subclass(Sub), False),      # a subclass may redefine what it is asked
            (new(40, 64).as_subclass(Sub), new(40, 64), False),
            (new(2048)[16:], new(2032), True),                       # a view with an offset
            (new(40, 64), None, True), (leaf, new(40, 64), True), (param, new(2049), True)]


def _with_grads(forms):
    params = []
    for p, g, _ in forms:
        if g is not None and g.dtype != p.dtype:
            p.grad_dtype = None  # a gradient of another dtype may be assigned
        p.grad = g
        params.append(p)
    return params


def test_what_bind_takes():
    forms = _gradient_forms("cpu")
    params = _with_grads(forms)
    handles = _handles(params)
    held, rest = _torch_face.bind(params, C.addressof(handles), len(handles))
    assert rest == [i for i, (_, _, taken) in enumerate(forms) if not taken]
    with BaseTorchFunctionMode():
        assert _torch_face.bind(params, C.addressof(handles), len(handles))[1] == list(range(len(params)))
    product = params[10] * 2  # not a leaf: asking for its gradient warns, in Python code
    assert _torch_face.bind([product], C.addressof(handles), len(handles))[1] == [0]
    assert _torch_face.bind([torch.empty(0)], C.addressof(handles), len(handles))[1] == [0]  # no address: the C call refuses it by name
    with pytest.raises(TypeError):
        _torch_face.bind(tuple(params), C.addressof(handles), len(handles))
    with pytest.raises(IndexError):  # a list that has grown since the optimizer was made
        _torch_face.bind(params + [torch.zeros(8)], C.addressof(handles), len(handles))
    for h in handles:
        L.lib().eri_param_release(h)


def test_what_update_many_leaves_to_python():
    a, g = torch.zeros(8), torch.zeros(8)
    leave = [({}, {}), ({"a": a}, {"b": g}), ({"a": a.double()}, {"a": g}), ({"a": a}, {"a": g.bfloat16()}),
             ({"a": torch.zeros(4, 4).t()[1:]}, {"a": torch.zeros(3, 4)}), ({"a": a}, {"a": torch.zeros(16)[::2]}),
             ({"a": a.as_subclass(Sub)}, {"a": g}), ({3: a}, {3: g}), ({"a": a.to_sparse()}, {"a": g})]
    for params, grads in leave:
        assert _torch_face.update_many(1, params, grads) is None
    with BaseTorchFunctionMode():
        assert _torch_face.update_many(1, {"a": a}, {"a": g}) is None


class _MadeOfTwo:
    """Parameters whose handles were made for 40 x 64 float32 elements."""

    def __init__(self):
        from eridiffusion_amd.adam8bit import _Made
        self.handles = _handles([torch.zeros(40, 64), torch.zeros(40, 64)])
        self.made = (_Made * 2)(_Made(2560, L.DTYPE_F32), _Made(2560, L.DTYPE_F32))

    def rest(self, *params):
        return _torch_face.bind(list(params), C.addressof(self.handles), 2, C.addressof(self.made))[1]


def test_bind_leaves_alone_what_a_kernel_would_overrun():
    """A launch is sized by what the optimizer was made for: smaller data, another dtype, a gradient that no longer has
    the parameter's size, and host memory stay out of it."""
    two = _MadeOfTwo()
    assert two.rest(torch.zeros(40, 64), torch.zeros(40, 64)) == [0, 1]  # ordinary host memory
    small, wide = torch.zeros(40, 64), torch.zeros(40, 64)
    small.data, wide.data = torch.zeros(16), torch.zeros(40, 64, dtype=torch.bfloat16)
    assert two.rest(small, wide) == [0, 1]
    shrunk = torch.zeros(40, 64, requires_grad=True)
    shrunk.grad = torch.zeros(40, 64)
    shrunk.grad.data = torch.zeros(16)
    assert _torch_face.bind([shrunk], C.addressof(two.handles), 2)[1] == [0]
    for h in two.handles:
        L.lib().eri_param_release(h)


def test_python_loops_refuse_what_a_kernel_would_overrun(monkeypatch):
    """No launch is queued for any of these; on a device the first two are faults."""
    from eridiffusion_amd import adam8bit
    monkeypatch.setattr(adam8bit, "_stream_ptr", lambda: 0)
    a, b = torch.zeros(4096), torch.zeros(16)
    assert _torch_face.update_many(1, {"a": a}, {"a": a}) is None
    opt = adam8bit.Adam8bitFunctional()
    for call in (lambda p, g: opt.update("a", p, g), lambda p, g: opt.update_many({"a": p}, {"a": g})):
        with pytest.raises(ValueError, match="device tensors"):
            call(a, a)
    with pytest.raises(ValueError, match="16 elements for a parameter of 4096"):
        adam8bit._usable_grad(b, a)
    with pytest.raises(ValueError, match="cannot read"):
        adam8bit._usable_grad(a, a)
    with pytest.raises(ValueError, match="moments of 4096 and 16"):
        opt.load_state_from_tensors({"a": (a, b)})
    lists = adam8bit.Adam8bit([torch.zeros(4096), torch.zeros(4096)])
    lists.params[0].grad = torch.zeros(4096)
    with pytest.raises(ValueError, match="host memory"):
        lists.step()
    for data, message in ((b, "16 elements"), (a.bfloat16(), "bfloat16"), (b[:1].expand(4096), "contiguous")):
        lists = adam8bit.Adam8bit([torch.zeros(4096)])
        lists.params[0].data = data
        assert lists.step() == 1  # nothing to step: it is left alone
        lists.params[0].grad = data.clone()
        with pytest.raises(ValueError, match=message):
            lists.step()


@pytest.mark.gpu
def test_sizes_and_devices_are_looked_at_before_a_launch():
    from eridiffusion_amd.adam8bit import Adam8bit, Adam8bitConfig, Adam8bitFunctional
    p, g = torch.randn(4096, device="cuda"), torch.randn(4096, device="cuda") * 1e-3
    fn = Adam8bitFunctional.with_params(1e-3, 0.9, 0.999, 1e-8, 0.01)
    for bad in (g[:16], g.cpu()):
        for call in (lambda: fn.update_many({"a": p}, {"a": bad}), lambda: fn.update("a", p, bad)):
            with pytest.raises(ValueError):
                call()
    assert fn.get_state_as_tensors() == {}
    want = fn.update_many({"a": p}, {"a": g})["a"].clone()
    other = Adam8bitFunctional.with_params(1e-3, 0.9, 0.999, 1e-8, 0.01)
    assert torch.equal(other.update_many({"a": p}, {"a": g.cpu().pin_memory()})["a"], want)  # pinned memory is read where it is
    opt = Adam8bit([p.clone()], Adam8bitConfig(lr=1e-3))
    opt.params[0].data = p[:16].clone()
    opt.params[0].grad = g[:16].clone()
    with pytest.raises(ValueError):
        opt.step()


@pytest.mark.gpu
def test_native_and_python_loops_step_alike():
    from eridiffusion_amd.adam8bit import Adam8bit, Adam8bitConfig, Adam8bitFunctional, update_params_8bit
    results = []
    for general in (False, True):
        forms = _gradient_forms("cuda")
        params = _with_grads(forms)
        opt = Adam8bit(params, Adam8bitConfig(lr=1e-3))
        for _ in range(2):
            if general:
                with BaseTorchFunctionMode():
                    assert opt.step() == 1
            else:
                assert opt.step() == 1
        named = {"t%d" % i: p.detach().clone() for i, (p, g, _) in enumerate(forms) if g is not None}
        grads = {"t%d" % i: g for i, (_, g, _) in enumerate(forms) if g is not None}
        plain = {n for i, (_, g, taken) in enumerate(forms) for n in ["t%d" % i] if taken and g is not None}
        outs = []
        for keep in (plain, set(named)):  # the plain ones alone take the native loop, all together the Python one
            fn = Adam8bitFunctional.with_params(1e-3, 0.9, 0.999, 1e-8, 0.01)
            now = {n: t for n, t in named.items() if n in keep}
            for _ in range(2):
                if general:
                    with BaseTorchFunctionMode():
                        update_params_8bit(fn, now, grads)
                else:
                    update_params_8bit(fn, now, grads)
                fn.step()
            assert list(fn.get_state_as_tensors()) == list(now)
            outs += [t.clone() for t in now.values()]
        torch.cuda.synchronize()
        results.append([p.detach().clone() for p in params] + outs)
    for a, b in zip(*results):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.gpu
def test_update_many_refusals_keep_their_codes():
    from eridiffusion_amd.adam8bit import Adam8bitFunctional
    fn = Adam8bitFunctional.with_params(1e-3, 0.9, 0.999, 1e-8, 0.01)
    fn.update_many({"a": torch.zeros(64, device="cuda")}, {"a": torch.zeros(64, device="cuda")})
    with pytest.raises(L.EriError) as e:  # a state of another size under the same name
        fn.update_many({"a": torch.zeros(128, device="cuda")}, {"a": torch.zeros(128, device="cuda")})
    assert e.value.code == -6
    with pytest.raises(L.EriError) as e:
        fn.update_many({"b": torch.zeros(0, device="cuda")}, {"b": torch.zeros(0, device="cuda")})
    assert e.value.code in (-1, -3)
    assert list(fn.get_state_as_tensors()) == ["a"]


def test_moments_loaded_under_another_stream_are_waited_for(monkeypatch):
    """Before they are read, and before the call lets go of them; on the optimizer's own stream nothing waits."""
    from eridiffusion_amd import adam8bit
    calls, stream = [], [11]

    class Lib:
        def __getattr__(self, name):
            return lambda *args: calls.append((name, args[0])) or 0
    monkeypatch.setattr(adam8bit, "lib", lambda: Lib())
    monkeypatch.setattr(adam8bit, "_stream_ptr", lambda: stream[0])
    opt = adam8bit.Adam8bitFunctional()
    del calls[:]
    state = {"a": (torch.zeros(8), torch.zeros(8)), "b": (torch.zeros(8), torch.zeros(8))}
    opt.load_state_from_tensors(state)
    assert [name for name, _ in calls] == ["eri_adam8bit_fn_load_state_fp32"] * 2
    del calls[:]
    stream[0] = 12
    opt.load_state_from_tensors(state)
    assert [(name, args) for name, args in calls if "sync" in name] == [("eri_hip_stream_sync", 12), ("eri_hip_stream_sync", 11)] * 2
    assert [name.endswith("fp32") for name, _ in calls] == [False, True, False] * 2


def test_moments_of_different_sizes_are_refused_before_any_is_loaded(monkeypatch):
    from eridiffusion_amd import adam8bit
    calls = []

    class Lib:
        def __getattr__(self, name):
            return lambda *args: calls.append(name) or 0
    monkeypatch.setattr(adam8bit, "lib", lambda: Lib())
    monkeypatch.setattr(adam8bit, "_stream_ptr", lambda: 11)
    opt = adam8bit.Adam8bitFunctional()
    del calls[:]
    with pytest.raises(ValueError, match="8 and 9 elements for 'b'"):
        opt.load_state_from_tensors({"a": (torch.zeros(8), torch.zeros(8)), "b": (torch.zeros(8), torch.zeros(9))})
    assert calls == [] and not opt._names


@pytest.mark.gpu
def test_names_are_loaded_in_the_order_of_the_dict():
    """Moments that are converted on the way between moments that are read as they are."""
    from eridiffusion_amd.adam8bit import Adam8bitFunctional
    state = {name: (torch.rand(3000, device="cuda").to(dt), torch.rand(3000, device="cuda").to(dt))
             for name, dt in (("d", torch.float32), ("a", torch.float64), ("c", torch.float32), ("e", torch.bfloat16), ("b", torch.float32))}
    opt = Adam8bitFunctional()
    opt.load_state_from_tensors(state)
    assert list(opt.get_state_as_tensors()) == list(state)
    for name, (m, v) in state.items():
        one = Adam8bitFunctional()
        one.load_state_from_tensors({name: (m.float(), v.float())})
        for a, b in zip(one.get_state_as_tensors()[name], opt.get_state_as_tensors()[name]):
            assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("pooled", [False, True])
def test_reload_under_another_stream(pooled):
    """Moments that a side stream is still making when they are loaded, float64 so that they are converted on the way,
    and whose memory that stream hands out and overwrites right behind the call."""
    from eridiffusion_amd.adam8bit import Adam8bitFunctional, DevicePool
    n = (1 << 22) + 5
    want, opt = Adam8bitFunctional(), Adam8bitFunctional()
    if pooled:
        opt.set_state_pool(DevicePool(64 << 20, 1), 0)
    m, v = torch.randn(n, device="cuda"), torch.rand(n, device="cuda")
    want.load_state_from_tensors({"w": (m, v)})
    opt.load_state_from_tensors({"w": (v, m.square())})
    busy = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for _ in range(8):
            busy = busy @ busy * 1e-2
        opt.load_state_from_tensors({"w": (m.double(), v.double())})
        trash = [torch.full((n,), 9.0, device="cuda") for _ in range(6)]
    torch.cuda.synchronize()
    for a, b in zip(opt.get_state_as_tensors()["w"], want.get_state_as_tensors()["w"]):
        assert torch.equal(a, b)
    assert len(trash) == 6


@pytest.mark.gpu
def test_out_of_memory_for_the_outputs_is_torchs_own_exception():
    from eridiffusion_amd.adam8bit import Adam8bitFunctional
    n = 1 << 25
    p, g = torch.randn(n, device="cuda"), torch.randn(n, device="cuda")
    fn = Adam8bitFunctional.with_params(1e-3, 0.9, 0.999, 1e-8, 0.01)
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            fn.update_many({"w": p}, {"w": g})
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert fn.get_state_as_tensors() == {} and fn.memory_stats() == (0, 0)
    assert fn.update_many({"w": p}, {"w": g})["w"].shape == p.shape


def test_a_closed_optimizer_answers_as_the_library_does(monkeypatch):
    from eridiffusion_amd import adam8bit
    monkeypatch.setattr(adam8bit, "_stream_ptr", lambda: 0)
    opt = adam8bit.Adam8bitFunctional()
    opt.close()
    with pytest.raises(L.EriError) as e:
        opt.update_many({}, {})
    assert e.value.code == -1


@pytest.mark.gpu
def test_outputs_of_named_updates_are_torchs_own():
    """Storages of their own on the parameter's device, seen by the allocator's counters and by a dispatch mode, and
    inference tensors under inference mode."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from eridiffusion_amd.adam8bit import Adam8bitFunctional
    fn = Adam8bitFunctional.with_params(1e-3, 0.9, 0.999, 1e-8, 0.01)
    params = {"a": torch.randn(40, 64, device="cuda"), "b": torch.randn(2049, device="cuda").to(torch.bfloat16)}
    grads = {k: torch.randn_like(v) for k, v in params.items()}
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    outs = fn.update_many(params, grads)
    assert torch.cuda.memory_stats()["allocation.all.allocated"] - before >= 2
    for k, v in outs.items():
        assert type(v) is torch.Tensor and v.shape == params[k].shape and v.dtype == params[k].dtype and v.device == params[k].device
        assert v.untyped_storage().nbytes() == v.numel() * v.element_size() and v.is_leaf and not v.requires_grad
    assert outs["a"].untyped_storage().data_ptr() != outs["b"].untyped_storage().data_ptr()

    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))
    with Mode():
        fn.update_many(params, grads)
    assert sum("empty" in s for s in seen) == 2
    with torch.inference_mode():
        assert all(v.is_inference() for v in fn.update_many(params, grads).values())
