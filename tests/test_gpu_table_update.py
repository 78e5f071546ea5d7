"""eri_adam8_table_update to new addresses: as many rows as a launch carries, one more, as many as two do and one more (a
copy of the rows), gradients alone and everything a step is given; against a table made at those addresses, bit for bit."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu
BLOCK = 2048


def _rows(sizes, layouts, p, g, state, p_src=None, scale=1.0):
    from eridiffusion_amd import _lib as L
    rows, at, blocks = (L.TensorRow * len(sizes))(), 0, 0
    m, v, am, av = state
    for r, n, layout in zip(rows, sizes, layouts):
        r.p, r.g, r.m, r.v = p.data_ptr() + 4 * at, g.data_ptr() + 4 * at, m.data_ptr() + at, v.data_ptr() + at
        if p_src is not None:
            r.p_src = p_src.data_ptr() + 4 * at
        r.absmax_m, r.absmax_v = am.data_ptr() + 4 * blocks, av.data_ptr() + 4 * blocks
        r.numel, r.block_start, r.grad_scale = n, blocks, scale
        r.dtype_tag, r.grad_f32 = (L.DTYPE_F32 if layout == 0 else L.DTYPE_BF16), int(layout == 2)
        at += (n + 15) // 16 * 16
        blocks += (n + BLOCK - 1) // BLOCK
    return rows


@pytest.mark.parametrize("what,n", [("addresses", k) for k in (1, 160, 161, 320, 321)] + [("gradients", k) for k in (480, 481, 960, 961)] + [("scale", 3)])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("other_stream", [False, True])
def test_rows_at_new_addresses(what, n, mixed, other_stream):
    import torch
    from eridiffusion_amd import _lib as L
    sizes = [1 + (i * 37) % 90 if i % 5 else 2050 for i in range(n)]
    layouts = [i % 3 if mixed else 1 for i in range(n)]
    total = sum((k + 15) // 16 * 16 for k in sizes)
    blocks = sum((k + BLOCK - 1) // BLOCK for k in sizes)
    gen = torch.Generator(device="cuda").manual_seed(n)

    def words(std):  # read as fp32 or, two to a word, as bf16
        return (torch.randn(2 * total, device="cuda", generator=gen) * std).to(torch.bfloat16)
    ps, gs = [words(0.02) for _ in range(2)], [words(1e-3) for _ in range(2)]
    main = torch.cuda.current_stream()
    h = L.hyper_pack(1e-3, 0.9, 0.999, 1e-8, 0.01, 1, L.MODE_ERI, L.FLAG_EXACT_PARAM)

    def state():
        s = (torch.empty(total, dtype=torch.uint8, device="cuda"), torch.empty(total, dtype=torch.uint8, device="cuda"),
             torch.empty(blocks, device="cuda"), torch.empty(blocks, device="cuda"))
        L.check(L.lib().eri_adam8_state_init(s[0].data_ptr(), s[1].data_ptr(), s[2].data_ptr(), s[3].data_ptr(), total, main.cuda_stream), "init")
        s[2].zero_(), s[3].zero_()
        return s

    def run(update):
        s, p, q = state(), ps[0].clone(), ps[1].clone()
        new = {"addresses": dict(p=q, g=gs[1], p_src=p), "gradients": dict(p=p, g=gs[1]), "scale": dict(p=p, g=gs[1], scale=0.5)}[what]
        table = C.c_void_p()
        first = _rows(sizes, layouts, p, gs[0], s) if update else _rows(sizes, layouts, state=s, **new)
        L.check(L.lib().eri_adam8_table_create(first, n, main.cuda_stream, C.byref(table)), "create")
        side = torch.cuda.Stream() if other_stream else main
        side.wait_stream(main)
        if update:
            L.check(L.lib().eri_adam8_table_update(table, _rows(sizes, layouts, state=s, **new), n, main.cuda_stream), "update")
        for _ in range(2):
            L.check(L.lib().eri_adam8_step_table(table, C.byref(h), side.cuda_stream), "step")
        torch.cuda.synchronize()
        L.lib().eri_adam8_table_destroy(table)
        return (p, q) + s

    for a, b in zip(run(True), run(False)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def _one(case, rows, k, stream):
    from eridiffusion_amd import _lib as L
    L.check(L.lib().eri_adam8_table_update(case, rows[k], len(rows[k]), stream.cuda_stream), "update")


@pytest.mark.parametrize("how", ["two_streams", "captured", "before_a_capture"])
def test_updates_follow_each_other(how):
    """Rows of a stream's update stay behind those of a later one on another; an update that a graph holds leaves the next
    one everything to set; and one in front of a capture on another stream is what the graph steps on."""
    import torch
    from eridiffusion_amd import _lib as L
    n, size = 40, 3000
    main, side = torch.cuda.current_stream(), torch.cuda.Stream()
    gen = torch.Generator(device="cuda").manual_seed(5)
    total, blocks = n * ((size + 15) // 16 * 16), n * 2
    ps = [torch.randn(2 * total, device="cuda", generator=gen).to(torch.bfloat16) for _ in range(2)]
    gs = [torch.randn(2 * total, device="cuda", generator=gen).to(torch.bfloat16) for _ in range(3)]
    h = L.hyper_pack(1e-3, 0.9, 0.999, 1e-8, 0.01, 1, L.MODE_ERI, L.FLAG_EXACT_PARAM)

    def run(update):
        s = (torch.zeros(total, dtype=torch.uint8, device="cuda"), torch.zeros(total, dtype=torch.uint8, device="cuda"),
             torch.zeros(blocks, device="cuda"), torch.zeros(blocks, device="cuda"))
        for i in range(n):
            at = i * ((size + 15) // 16 * 16)
            L.check(L.lib().eri_adam8_state_init(s[0].data_ptr() + at, s[1].data_ptr() + at, s[2].data_ptr() + 8 * i, s[3].data_ptr() + 8 * i,
                                                 size, main.cuda_stream), "init")
        p = [x.clone() for x in ps]
        rows = [_rows([size] * n, [1] * n, p[a], gs[b], s) for a, b in ((0, 0), (1, 1), (1, 2))]
        table, last = C.c_void_p(), 2 if how != "before_a_capture" else 1
        L.check(L.lib().eri_adam8_table_create(rows[0 if update else last], n, main.cuda_stream, C.byref(table)), "create")

        def step(stream):
            L.check(L.lib().eri_adam8_step_table(table, C.byref(h), stream.cuda_stream), "step")
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        if how == "two_streams":
            if update:
                _one(table, rows, 0, main)
                torch.cuda._sleep(20_000_000)
                _one(table, rows, 1, main)
                _one(table, rows, 2, side)
            step(side)
            torch.cuda.synchronize()
            step(side)
        elif how == "captured":
            if update:
                with torch.cuda.graph(graph):
                    _one(table, rows, 1, torch.cuda.current_stream())
                _one(table, rows, 2, main)
            step(main)
            step(main)
        else:
            if update:
                _one(table, rows, 1, main)
                with torch.cuda.graph(graph):
                    step(torch.cuda.current_stream())
                for _ in range(2):
                    graph.replay()
                    torch.cuda.synchronize()
            else:
                step(main)
                step(main)
        torch.cuda.synchronize()
        L.lib().eri_adam8_table_destroy(table)
        return tuple(p) + s

    for a, b in zip(run(True), run(False)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
