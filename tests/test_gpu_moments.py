"""The kernels between fp32 moments and codes + absmax at the sizes and addresses where they can go wrong: remainders of
the four elements a lane holds, of a 256-element pass and of a block, whole words and single elements, negative
values under the unsigned map.  The format is specified bit for bit: every comparison is exact."""
import numpy as np
import pytest

import harness as hs
import oracle_c as oc

pytestmark = pytest.mark.gpu


def _moments(n, signed, rng):
    x = (rng.standard_normal(n) * 10.0 ** rng.uniform(-6, 0, n)).astype(np.float32)
    x[rng.random(n) < 0.05] = 0.0  # negative values stay in for the unsigned map too: they take code 0
    return x


@pytest.mark.parametrize("n", [1, 3, 4, 5, 255, 257, 2047, 2048, 2049, 4099, 3 * 2048 + 1022, 2048 * 4100 + 7])
@pytest.mark.parametrize("x_off,code_off", [(0, 0), (1, 0), (0, 1), (4, 4)])
def test_quantise_and_dequantise_equal_the_oracle(n, x_off, code_off):
    import torch
    from eridiffusion_amd import _lib as L
    rng = np.random.default_rng(n + 7 * x_off + code_off)
    nb = (n + 2047) // 2048
    dev, stream = torch.device("cuda:0"), torch.cuda.current_stream().cuda_stream
    guard = 64
    xs, want = [], []
    for signed in (1, 0):
        x = _moments(n, signed, rng)
        wc, wa, wb = np.empty(n, np.uint8), np.empty(nb, np.float32), np.empty(n, np.float32)
        oc.lib().eri_oracle_quantize(oc.ptr(x), oc.ptr(hs.MAPS[1 - signed]), n, oc.ptr(wc), oc.ptr(wa))
        oc.lib().eri_oracle_dequantize(oc.ptr(wc), oc.ptr(wa), oc.ptr(hs.MAPS[1 - signed]), n, oc.ptr(wb))
        xs.append(x)
        want.append((wc, wa, wb))

    def buffers():
        xd = [torch.full((n + x_off + guard,), 7.0, device=dev) for _ in xs]
        for d, x in zip(xd, xs):
            d[x_off:x_off + n] = torch.from_numpy(x).to(dev)
        codes = [torch.full((n + code_off + guard,), 99, dtype=torch.uint8, device=dev) for _ in xs]
        absmax = [torch.full((nb + guard,), 5.0, device=dev) for _ in xs]
        back = [torch.full((n + x_off + guard,), 7.0, device=dev) for _ in xs]
        return xd, codes, absmax, back

    def check(codes, absmax, back):
        torch.cuda.synchronize()
        for i in (0, 1):
            c, a, b = codes[i].cpu().numpy(), absmax[i].cpu().numpy(), back[i].cpu().numpy()
            wc, wa, wb = want[i]
            assert np.array_equal(c[code_off:code_off + n], wc), i
            assert np.array_equal(a[:nb].view(np.uint32), wa.view(np.uint32)), i
            assert np.array_equal(b[x_off:x_off + n].view(np.uint32), wb.view(np.uint32)), i
            assert (c[:code_off] == 99).all() and (c[code_off + n:] == 99).all(), i  # nothing outside the tensor is written
            assert (a[nb:] == 5.0).all() and (b[:x_off] == 7.0).all() and (b[x_off + n:] == 7.0).all(), i

    xd, codes, absmax, back = buffers()
    x_ptr = [d.data_ptr() + 4 * x_off for d in xd]
    c_ptr = [c.data_ptr() + code_off for c in codes]
    b_ptr = [b.data_ptr() + 4 * x_off for b in back]
    for i, signed in enumerate((1, 0)):
        L.check(L.lib().eri_adam8_quantize(x_ptr[i], signed, n, c_ptr[i], absmax[i].data_ptr(), stream), "quantize")
        L.check(L.lib().eri_adam8_dequantize(c_ptr[i], absmax[i].data_ptr(), signed, n, b_ptr[i], stream), "dequantize")
    check(codes, absmax, back)

    xd, codes, absmax, back = buffers()  # both moments in one launch
    x_ptr = [d.data_ptr() + 4 * x_off for d in xd]
    c_ptr = [c.data_ptr() + code_off for c in codes]
    b_ptr = [b.data_ptr() + 4 * x_off for b in back]
    am, av = absmax[0].data_ptr(), absmax[1].data_ptr()
    L.check(L.lib().eri_adam8_quantize_state(x_ptr[0], x_ptr[1], n, c_ptr[0], c_ptr[1], am, av, stream), "quantize_state")
    L.check(L.lib().eri_adam8_dequantize_state(c_ptr[0], c_ptr[1], am, av, n, b_ptr[0], b_ptr[1], stream), "dequantize_state")
    check(codes, absmax, back)


def test_loading_moments_of_the_same_size_keeps_the_state_where_it_is():
    """update, load, update: the second update starts from the loaded moments, and a load that is refused (the second
    moment is ordinary host memory) leaves the state as it was."""
    import torch
    from eridiffusion_amd import _lib as L
    from eridiffusion_amd.adam8bit import Adam8bitFunctional
    n = 2048 * 3 + 130
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(11)
    p, g = torch.randn(n, device=dev, generator=gen), torch.randn(n, device=dev, generator=gen) * 1e-3
    m, v = torch.randn(n, device=dev, generator=gen) * 1e-3, torch.rand(n, device=dev, generator=gen) * 1e-6
    used, new = Adam8bitFunctional(), Adam8bitFunctional()
    used.update("w", p, g)
    used.load_state_from_tensors({"w": (m, v)})
    new.load_state_from_tensors({"w": (m, v)})
    assert torch.equal(used.update("w", p, g), new.update("w", p, g))
    before = used.get_state_as_tensors()["w"]
    host = np.zeros(n, np.float32)
    assert L.lib().eri_adam8bit_fn_load_state_fp32(used._opt, b"w", p.data_ptr(), host.ctypes.data, n) == -6
    after = used.get_state_as_tensors()["w"]
    assert torch.equal(before[0], after[0]) and torch.equal(before[1], after[1])


@pytest.mark.parametrize("names", [3, 48, 49, 130])
@pytest.mark.parametrize("pooled", [False, True])
def test_many_states_in_one_call(names, pooled):
    """Fewer tensors than one launch takes, as many, one more, and three launches; sizes around the four blocks of a
    workgroup, one pair of moments at an odd address; against the same calls name by name, bit for bit, on an optimizer
    that has the states already and on one that makes them."""
    import torch
    from eridiffusion_amd.adam8bit import Adam8bitFunctional, DevicePool
    gen = torch.Generator(device="cuda").manual_seed(names)
    sizes = [(5, 2047, 2048, 2049, 4 * 2048, 4 * 2048 + 1, 8 * 2048 - 3)[i % 7] + 3 * i for i in range(names)]
    state = {"n%d" % i: (torch.randn(n, device="cuda", generator=gen) * 1e-3, torch.rand(n, device="cuda", generator=gen) * 1e-6)
             for i, n in enumerate(sizes)}
    state["n1"] = tuple(torch.cat([x.new_zeros(1), x])[1:] for x in state["n1"])
    one, many = Adam8bitFunctional(), Adam8bitFunctional()
    if pooled:
        many.set_state_pool(DevicePool(64 << 20, 1), 0)
    for name, moments in state.items():
        one.load_state_from_tensors({name: moments})
    for _ in range(2):
        many.load_state_from_tensors(state)
        a, b = one.get_state_as_tensors(), many.get_state_as_tensors()
        assert list(a) == list(b) == list(state)
        for name in state:
            assert torch.equal(a[name][0], b[name][0]) and torch.equal(a[name][1], b[name][1]), name


def test_a_name_twice_in_one_load_keeps_its_last_contents():
    import ctypes as C
    import torch
    from eridiffusion_amd import _lib as L
    from eridiffusion_amd.adam8bit import Adam8bitFunctional
    n = 5000
    gen = torch.Generator(device="cuda").manual_seed(3)
    xs = [torch.rand(n, device="cuda", generator=gen) for _ in range(6)]
    opt, want = Adam8bitFunctional(), Adam8bitFunctional()
    names = (C.c_char_p * 3)(b"a", b"b", b"a")
    ptr = [(C.c_void_p * 3)(*[x.data_ptr() for x in xs[k::2]]) for k in (0, 1)]
    for _ in range(2):  # states that the call makes, then states that are there
        L.check(L.lib().eri_adam8bit_fn_load_states_fp32(opt._opt, names, ptr[0], ptr[1], (C.c_uint64 * 3)(n, n, n), 3), "load")
        opt._names.update({"a": None, "b": None})
        want.load_state_from_tensors({"a": (xs[4], xs[5]), "b": (xs[2], xs[3])})
        for name, moments in want.get_state_as_tensors().items():
            assert all(torch.equal(x, y) for x, y in zip(opt.get_state_as_tensors()[name], moments)), name
    out = torch.empty(n, device="cuda")
    unknown = (C.c_void_p * 2)(out.data_ptr(), out.data_ptr())
    out.fill_(5.0)
    assert L.lib().eri_adam8bit_fn_get_states_fp32(opt._opt, (C.c_char_p * 2)(b"a", b"nobody"), unknown, unknown, 2) == -6
    assert bool((out == 5.0).all())  # nothing of a refused call runs


def _load_many(opt, rows):
    """rows: (name, m, v, numel) of eri_adam8bit_fn_load_states_fp32; addresses or tensors."""
    import ctypes as C
    from eridiffusion_amd import _lib as L
    k = len(rows)
    at = lambda x: x if isinstance(x, int) else x.data_ptr()
    return L.lib().eri_adam8bit_fn_load_states_fp32(opt._opt, (C.c_char_p * k)(*[r[0].encode() for r in rows]), (C.c_void_p * k)(*[at(r[1]) for r in rows]),
                                                    (C.c_void_p * k)(*[at(r[2]) for r in rows]), (C.c_uint64 * k)(*[r[3] for r in rows]), k)


def test_a_load_refused_behind_a_repeated_name_converts_nothing():
    import torch
    from eridiffusion_amd.adam8bit import Adam8bitFunctional
    n = 3000
    x = [torch.rand(n, device="cuda") for _ in range(3)]
    opt = Adam8bitFunctional()
    opt.load_state_from_tensors({"a": (x[0], x[0])})
    before = opt.get_state_as_tensors()["a"]
    host = np.ones(n, dtype=np.float32)
    assert _load_many(opt, [("a", x[1], x[1], n), ("b", x[2], x[2], n), ("a", x[2], x[2], n), ("c", x[1], host.ctypes.data, n)]) == -6
    after = opt.get_state_as_tensors()["a"]
    assert torch.equal(before[0], after[0]) and torch.equal(before[1], after[1])
    assert opt.memory_stats()[0] == 1


def test_a_failed_load_leaves_no_marks_for_the_next_updates():
    """Memory runs out behind names that exist: the update of these names is one launch, as before."""
    import ctypes as C
    import torch
    from eridiffusion_amd import _lib as L
    from eridiffusion_amd.adam8bit import Adam8bitFunctional, DevicePool
    n = 5000
    opt = Adam8bitFunctional()
    opt.set_state_pool(DevicePool(2 << 20, 1), 0)
    x = torch.rand(8 << 20, device="cuda")
    state = {name: (x[:n], x[:n]) for name in ("a", "b", "c")}
    opt.load_state_from_tensors(state)
    params = {k: torch.randn(n, device="cuda").to(torch.bfloat16) for k in state}
    grads = {k: torch.randn_like(v) for k, v in params.items()}
    opt.update_many(params, grads)
    assert _load_many(opt, [(k, x, x, n) for k in state] + [("large", x, x, x.numel())]) != 0

    def flushes():
        f, u = C.c_uint64(), C.c_uint64()
        L.check(L.lib().eri_adam8bit_fn_table_stats(opt._opt, C.byref(f), C.byref(u)), "table_stats")
        return f.value
    before = flushes()
    opt.update_many(params, grads)
    assert flushes() == before + 1


def test_loading_many_new_names_takes_time_by_their_number():
    import time
    import torch
    from eridiffusion_amd.adam8bit import Adam8bitFunctional, DevicePool
    x, times = torch.rand(64, device="cuda"), {}
    for k in (2000, 2000, 16000, 2000, 16000):  # the shorter of the two each; the first for warm-up
        opt = Adam8bitFunctional()
        opt.set_state_pool(DevicePool(32 << 20, 1), 0)
        rows = [("lora_unet_down_blocks_1_attentions_0_transformer_blocks_0_attn1_to_q.lora_down.weight.%d" % i, x, x, 64) for i in range(k)]
        torch.cuda.synchronize()
        start = time.perf_counter()
        assert _load_many(opt, rows) == 0
        times[k] = min(times.get(k, 1e9), time.perf_counter() - start)
    assert times[16000] < 14 * times[2000], times  # eight times as many names; 30 with a search through those before


def test_states_of_other_sizes_take_the_room_of_those_they_replace():
    """A lane that holds all states and one more (a piece goes to states of its size again), loaded with the sizes of
    neighbours exchanged: name by name that fits."""
    import torch
    from eridiffusion_amd.adam8bit import Adam8bitFunctional, DevicePool
    gen = torch.Generator(device="cuda").manual_seed(11)

    def moments(sizes):
        return {"w%d" % i: (torch.randn(n, device="cuda", generator=gen) * 1e-3, torch.rand(n, device="cuda", generator=gen) * 1e-6)
                for i, n in enumerate(sizes)}
    first, second = moments([200_000, 190_001] * 4), moments([190_001, 200_000] * 4)
    tight, roomy = Adam8bitFunctional(), Adam8bitFunctional()
    tight.set_state_pool(DevicePool(4 << 20, 1), 0)  # eight states take 3.1 MB
    for opt in (tight, roomy):
        opt.load_state_from_tensors(first)
        opt.load_state_from_tensors(second)
    a, b = tight.get_state_as_tensors(), roomy.get_state_as_tensors()
    for name in second:
        assert torch.equal(a[name][0], b[name][0]) and torch.equal(a[name][1], b[name][1]), name


def test_a_load_holds_little_of_what_it_replaces():
    """Twelve states of 24 MiB made anew, as above: how far up their lane they reach says how many were held at once."""
    import torch
    from eridiffusion_amd.adam8bit import Adam8bitFunctional, DevicePool
    n, k = 12 << 20, 12
    x = torch.rand(n, device="cuda") * 1e-3
    opt, pool = Adam8bitFunctional(), DevicePool(1 << 30, 1)
    base = pool.alloc_ptr(0, 256)
    opt.set_state_pool(pool, 0)
    for turn in (0, 1):
        assert _load_many(opt, [("w%d" % i, x, x, n - 4096 * ((i + turn) % 2)) for i in range(k)]) == 0
    top = pool.alloc_ptr(0, k * 24 << 20) - base  # larger than any hole: behind the highest piece in use
    assert top < (k + 5) * 25 << 20


def test_one_moment_at_an_odd_address_leaves_the_others_of_its_call_as_fast():
    """Element by element a moment takes 1.6 times as long as in whole words; one of 24 at an odd address may add a 24th of
    that and a launch, not slow all of them down."""
    import torch
    from eridiffusion_amd.adam8bit import Adam8bitFunctional
    n, times = 4 << 20, {}
    for odd in (0, 1, 0, 1):
        opt, state = Adam8bitFunctional(), {}
        for i in range(24):
            at = odd if i == 5 else 0
            state["n%d" % i] = tuple(torch.rand(n + 1, device="cuda")[at:at + n] for _ in range(2))
        opt.load_state_from_tensors(state)
        for _ in range(10):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            opt.load_state_from_tensors(state)
            end.record()
            end.synchronize()
            times[odd] = min(times.get(odd, 1e9), start.elapsed_time(end))
        back = opt.get_state_as_tensors()
        for name, moments in state.items():
            alone = Adam8bitFunctional()
            alone.load_state_from_tensors({name: tuple(x.clone() for x in moments)})
            a = alone.get_state_as_tensors()[name]
            assert torch.equal(a[0], back[name][0]) and torch.equal(a[1], back[name][1]), name
    assert times[1] < 1.3 * times[0], times
