"""Launches whose workgroups take their rounds of blocks by ticket: lists that end at, just before and just behind a
round, fewer rounds than workgroups and more, and the same table launched again and again (the counter is back at zero
each time), against the oracle, bit for bit."""
import ctypes as C

import pytest

import harness as hs
import test_gpu_whole_tables as whole

pytestmark = pytest.mark.gpu
WAVES, UNITS = 8, 256


@pytest.mark.parametrize("bf16", [True, False], ids=["bf16", "f32"])
@pytest.mark.parametrize("blocks", [1, WAVES - 1, WAVES, WAVES + 1, 5 * WAVES, WAVES * UNITS - 1, WAVES * UNITS, WAVES * UNITS + 1, 2 * WAVES * UNITS + 3])
def test_step_by_ticket(bf16, blocks):
    import torch
    from eridiffusion_amd import _lib as L
    sizes = [n for n in ((blocks + 1) // 2 * 2048, blocks // 2 * 2048) if n] + [100]
    ps, gs = hs.make_inputs(sizes, bf16, blocks)
    states = hs.oracle_states(sizes)
    gt = hs.GpuTensors([p.copy() for p in ps], gs, states, bf16)
    rows, table = gt.rows(), C.c_void_p()
    L.check(L.lib().eri_adam8_table_create(rows, len(rows), None, C.byref(table)), "table_create")
    for step in (1, 2, 3):
        args = (1e-3, 0.9, 0.999, 1e-8, 0.01, step)
        hs.oracle_step(ps, gs, states, args, bf16)
        h = L.hyper_pack(*args, L.MODE_ERI, L.FLAG_EXACT_PARAM | L.FLAG_ONE_WAVE)
        L.check(L.lib().eri_adam8_step_table(table, C.byref(h), None), "step_table")
    torch.cuda.synchronize()
    got_p, got_st = gt.fetch()
    assert hs.compare(got_p, got_st, ps, states, bf16, True, "blocks %d" % blocks)["code_mismatch"] == 0
    L.lib().eri_adam8_table_destroy(table)


@pytest.mark.parametrize("dtype,master", [("bf16", False), ("bf16", True), ("f32", False)])
@pytest.mark.parametrize("extra", [1, 5, 4 * UNITS + 3])
def test_sweeps_by_ticket(dtype, master, extra):
    """The 32-bit step and the EMA over lists just longer than the small kernels take, against the small kernels over the
    same rows in two calls, bit for bit; twice, so that the counter has been put back once."""
    import torch
    from eridiffusion_amd import _lib as L
    line = 128 * UNITS
    halves = [[(line // 2 + extra) * 2048 + 1500, 700, 2048 * 2 + 3], [(line // 2) * 2048 - 2048 * 3 + 1027]]
    sizes = halves[0] + halves[1]
    dt, tag = (torch.bfloat16, L.DTYPE_BF16) if dtype == "bf16" else (torch.float32, L.DTYPE_F32)
    stream = torch.cuda.current_stream().cuda_stream

    def run(groups):
        gen = torch.Generator(device="cuda").manual_seed(extra)
        at, total = [], 0
        for n in sizes:
            at.append(total)
            total += (n + 15) // 16 * 16
        p, g = [(torch.randn(total, device="cuda", generator=gen) * s).to(dt) for s in (0.02, 1e-3)]
        m, v = torch.randn(total, device="cuda", generator=gen) * 1e-3, torch.rand(total, device="cuda", generator=gen) * 1e-6
        w, shadow = p.float() * 1.0001, p * 0.5
        for _ in range(2):
            for ids in groups:
                rows, ema = (L.AdamW32Row * len(ids))(), (L.EmaRow * len(ids))()
                for r, e, i in zip(rows, ema, ids):
                    o = at[i]
                    r.p, r.g, r.m, r.v = p[o:].data_ptr(), g[o:].data_ptr(), m[o:].data_ptr(), v[o:].data_ptr()
                    r.master = w[o:].data_ptr() if master else None
                    r.numel, r.dtype_tag = sizes[i], tag
                    e.shadow, e.p, e.numel, e.dtype_tag = shadow[o:].data_ptr(), p[o:].data_ptr(), sizes[i], tag
                h = L.AdamW32Hyper(1e-3, 0.9, 0.999, 1e-8, 0.01)
                L.check(L.lib().eri_adamw32_step_multi(rows, len(ids), C.byref(h), stream), "adamw32")
                L.check(L.lib().eri_ema_update_multi(ema, len(ids), 0.9, stream), "ema")
        torch.cuda.synchronize()
        return p, m, v, w, shadow

    for a, b in zip(run([[0, 1, 2, 3]]), run([[0, 1, 2], [3]])):
        assert torch.equal(a, b)


def test_probe_step_and_step_with_ema_share_a_counter():
    """In turn over one table, each with the rounds of its own; against the steps alone on the plain kernel, bit for bit."""
    import torch
    from test_gpu_graph_capture import _tensors
    from eridiffusion_amd import _lib as L
    sizes = [50 * UNITS * 2048 + 300, 2048, 77, 7 * 2048]
    ours, plain = _tensors(sizes, 9), _tensors(sizes, 9)
    stream = torch.cuda.current_stream().cuda_stream
    for step in (1, 2, 3):
        for flags in (L.FLAG_EMA, 0):
            for (table, _, _, _), named in ((ours, 0), (plain, L.FLAG_NO_PIPELINE)):
                if table is ours[0]:
                    L.check(L.lib().eri_adam8_traffic_probe(table, stream), "traffic_probe")
                h = L.hyper_pack(1e-3, 0.9, 0.999, 1e-8, 0.01, step, L.MODE_ERI, L.FLAG_EXACT_PARAM | flags | named)
                h.ema_decay = 0.9
                L.check(L.lib().eri_adam8_step_table(table, C.byref(h), stream), "step_table")
    torch.cuda.synchronize()
    for a, b in zip(ours[3], plain[3]):
        assert torch.equal(a, b)
    for tensors in (ours, plain):
        L.lib().eri_adam8_table_destroy(tensors[0])


def _sweep(what, dtype, sizes, parts):
    """The sweep over tensors of these sizes, in `parts` calls; what it leaves behind, and the shortest us of a pass."""
    import torch
    from eridiffusion_amd import _lib as L
    dt, tag = (torch.float32, L.DTYPE_F32) if dtype == "f32" else (torch.bfloat16, L.DTYPE_BF16)
    stream = torch.cuda.current_stream().cuda_stream
    at = [0]
    for n in sizes:
        at.append(at[-1] + (n + 15) // 16 * 16)
    gen = torch.Generator(device="cuda").manual_seed(len(sizes))
    p, g = [(torch.randn(at[-1], device="cuda", generator=gen) * s).to(dt) for s in (0.02, 1e-3)]
    m, v, w = torch.randn(at[-1], device="cuda", generator=gen) * 1e-3, torch.rand(at[-1], device="cuda", generator=gen) * 1e-6, p.float()
    calls = []
    for k in range(parts):
        ids = range(len(sizes) * k // parts, len(sizes) * (k + 1) // parts)
        rows = ((L.EmaRow if what == "ema" else L.AdamW32Row) * len(ids))()
        for r, i in zip(rows, ids):
            r.p, r.numel, r.dtype_tag = p.data_ptr() + at[i] * p.element_size(), sizes[i], tag
            if what == "ema":
                r.shadow = g.data_ptr() + at[i] * g.element_size()
            else:
                r.g, r.m, r.v = g.data_ptr() + at[i] * g.element_size(), m.data_ptr() + 4 * at[i], v.data_ptr() + 4 * at[i]
                r.master = w.data_ptr() + 4 * at[i] if dtype == "master" else None
        calls.append(rows)
    h, best = L.AdamW32Hyper(1e-3, 0.9, 0.999, 1e-8, 0.01), 1e9
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    for turn in range(4):
        torch.cuda._sleep(20_000_000)  # the calls are queued before the first of them starts
        ev[0].record()
        for rows in calls:
            if what == "ema":
                L.check(L.lib().eri_ema_update_multi(rows, len(rows), 0.9, stream), "ema")
            else:
                L.check(L.lib().eri_adamw32_step_multi(rows, len(rows), C.byref(h), stream), "adamw32")
        ev[1].record()
        ev[1].synchronize()
        if turn:  # the first uploads its rows
            best = min(best, ev[0].elapsed_time(ev[1]) * 1000)
    return (p, g, m, v, w), best


@pytest.mark.parametrize("what,dtype,size", [("ema", "bf16", 301), ("ema", "f32", 301), ("ema", "bf16", 1501), ("adamw32", "bf16", 301),
                                             ("adamw32", "master", 301), ("adamw32", "f32", 301)])
def test_long_sweeps_of_partial_blocks_take_no_longer_in_one_call(what, dtype, size):
    """40,000 tensors against twice 20,000, which take the small kernels by their number: 1.8 to 3.6 times as long on the
    persistent ones."""
    import torch
    (one, t_one), (two, t_two) = (_sweep(what, dtype, [size] * 40_000, parts) for parts in (1, 2))
    for a, b in zip(one, two):
        assert torch.equal(a, b)
    assert t_one < 1.4 * t_two, (t_one, t_two)


@pytest.mark.parametrize("what,dtype,per_tail", [("ema", "bf16", 2), ("ema", "f32", 1), ("adamw32", "bf16", 2), ("adamw32", "master", 1), ("adamw32", "f32", 1)])
@pytest.mark.parametrize("over", [-1, 0, 1])
def test_both_sides_of_the_line_for_sweeps_of_partial_blocks(what, dtype, per_tail, over):
    """`per_tail` full blocks to a partial one, and one block fewer and more, against the same tensors in two calls."""
    import torch
    sizes = [per_tail * 2048 + 1 + i * 13 % 2047 for i in range(22_000)] + [2048 * (1 + over)] * (over >= 0)
    if over < 0:
        sizes[0] -= 2048
    one, two = (_sweep(what, dtype, sizes, parts)[0] for parts in (1, 3))
    for a, b in zip(one, two):
        assert torch.equal(a, b)


LINES = {("bf16", 0): 48, ("bf16", 1): 96, ("bf16", 2): 128, ("bf16-f32-grads", 0): 48, ("bf16-f32-grads", 1): 48,
         ("bf16-f32-grads", 2): 56, ("f32", 0): 40, ("f32", 1): 48, ("f32", 2): 48}


@pytest.mark.parametrize("layout,mode", sorted(LINES), ids=str)
@pytest.mark.parametrize("over,tail", [(0, 0), (1, 0), (1, 515)])
def test_both_sides_of_the_line_to_the_prefetching_kernel(layout, mode, over, tail):
    """The dispatch's own choice just below and above, against the plain kernel, bit for bit."""
    import torch
    from eridiffusion_amd import _lib as L
    sizes = whole._sizes(LINES[layout, mode] * UNITS + over, tail)
    for a, b in zip(whole._run(layout, mode, sizes, 0, 0.5), whole._run(layout, mode, sizes, L.FLAG_NO_PIPELINE, 0.5)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("layout,mode", [("bf16", 0), ("bf16-f32-grads", 1), ("f32", 0)])
@pytest.mark.parametrize("long_tails", [-1, 0, 1])
def test_both_sides_of_the_line_for_long_partial_blocks(layout, mode, long_tails):
    """Just as many partial blocks of more than half a block as the prefetching kernel takes, one fewer and one more."""
    import torch
    from eridiffusion_amd import _lib as L
    full = LINES[layout, mode] * UNITS + 6
    tails = full // (3 if layout == "bf16" else 2) + long_tails
    sizes = [2048 + 1025 + i % 9 for i in range(tails)] + [(full - tails) * 2048 + 1024]
    for a, b in zip(whole._run(layout, mode, sizes, 0, 0.5), whole._run(layout, mode, sizes, L.FLAG_NO_PIPELINE, 0.5)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("layout,line", [("bf16", 24), ("bf16-f32-grads", 14)])
@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("tail", [0, 515])
def test_both_sides_of_the_line_to_the_step_that_carries_the_ema(layout, line, over, tail):
    import torch
    from eridiffusion_amd import _lib as L
    sizes = whole._sizes(line * UNITS + over, tail)
    for a, b in zip(whole._run(layout, 0, sizes, 0, None, ema=True), whole._run(layout, 0, sizes, L.FLAG_NO_PIPELINE, None, ema=True)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("mode", [0, 1, 2], ids=["eri", "l2", "bnb"])
@pytest.mark.parametrize("layout", ["bf16", "bf16-f32-grads", "f32"])
def test_partial_blocks_of_the_prefetching_kernel(layout, mode):
    """Parts that end in and on the edges of every pass of 512 elements, against the plain kernel, bit for bit."""
    import torch
    from eridiffusion_amd import _lib as L
    parts = [1, 7, 8, 505, 511, 512, 513, 1023, 1024, 1025, 1535, 1536, 1537, 2040, 2041, 2047]
    sizes = [(i % 3) * 2048 + n for i, n in enumerate(parts * 3)]
    for a, b in zip(whole._run(layout, mode, sizes, L.FLAG_ONE_WAVE, 0.5), whole._run(layout, mode, sizes, L.FLAG_NO_PIPELINE, 0.5)):
        assert torch.equal(a, b)


def _time_of(layout, mode, sizes, kinds):
    """Shortest us per launch of a table of these sizes for each of the kinds (flags, EMA)."""
    import torch
    from eridiffusion_amd import _lib as L
    stream = torch.cuda.current_stream().cuda_stream
    blocks = [(n + 2047) // 2048 for n in sizes]
    words = {"bf16": (2, 2), "bf16-f32-grads": (2, 4), "f32": (4, 4)}[layout]
    p, g = ((torch.randn(sum(blocks) * 2048, device="cuda") * 1e-3).to(torch.bfloat16 if w == 2 else torch.float32) for w in words)
    shadow, m, v = (torch.zeros(sum(blocks) * 2048 * w, dtype=torch.uint8, device="cuda") for w in (words[0], 1, 1))
    am, av = (torch.zeros(sum(blocks), device="cuda") for _ in range(2))
    rows, at = (L.TensorRow * len(sizes))(), 0
    for r, n, b in zip(rows, sizes, blocks):
        r.p, r.g, r.ema_shadow = p.data_ptr() + at * 2048 * words[0], g.data_ptr() + at * 2048 * words[1], shadow.data_ptr() + at * 2048 * words[0]
        r.m, r.v, r.absmax_m, r.absmax_v = m.data_ptr() + at * 2048, v.data_ptr() + at * 2048, am.data_ptr() + 4 * at, av.data_ptr() + 4 * at
        r.numel, r.block_start, r.grad_scale = n, at, 1.0
        r.dtype_tag, r.grad_f32 = (L.DTYPE_F32 if layout == "f32" else L.DTYPE_BF16), int(layout == "bf16-f32-grads")
        at += b
    table, best = C.c_void_p(), [1e9] * len(kinds)
    L.check(L.lib().eri_adam8_table_create(rows, len(rows), stream, C.byref(table)), "table_create")
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    for _ in range(5):
        for k, (flags, ema) in enumerate(kinds):
            h = L.hyper_pack(1e-3, 0.9, 0.999, 1e-8, 0.01, 3, mode, flags | (L.FLAG_EMA if ema else 0))
            h.ema_decay = 0.9
            ev[0].record()
            for _ in range(10):
                L.check(L.lib().eri_adam8_step_table(table, C.byref(h), stream), "step_table")
            ev[1].record()
            ev[1].synchronize()
            best[k] = min(best[k], ev[0].elapsed_time(ev[1]) * 100)
    L.lib().eri_adam8_table_destroy(table)
    return best


@pytest.mark.parametrize("layout,mode,size", [("bf16", 0, 4095), ("bf16", 1, 4095), ("bf16", 2, 3549), ("bf16-f32-grads", 1, 4095)])
def test_tables_of_many_partial_blocks_take_no_longer_than_on_the_plain_kernel(layout, mode, size):
    """As many partial blocks as full ones, behind the line: 1.4 to 1.7 times as long when the prefetching kernel went
    over the parts twice, a pass at a time, 1.1 to 1.2 times when it took them once."""
    from eridiffusion_amd import _lib as L
    ours, plain = _time_of(layout, mode, [size] * (140 * UNITS), [(0, False), (L.FLAG_NO_PIPELINE, False)])
    assert ours < 1.06 * plain, (ours, plain)
