"""The steady-state step allocates nothing and synchronises nothing, so a caller can capture it in a HIP
graph (useful for the launch-bound LoRA-sized workloads).  The graph holds the gradient-norm pass and the
step that consumes its clip factor; it is replayed several times with eager work and synchronisations in
between, and every replay is checked against the same sequence issued eagerly on a second copy."""
import ctypes as C

import numpy as np
import pytest

import harness as hs

pytestmark = pytest.mark.gpu
LR, B1, B2, EPS, WD = 1e-4, 0.9, 0.999, 1e-8, 0.01


@pytest.mark.parametrize("bf16", [True, False])
def test_graph_replays_equal_eager_steps(bf16):
    import torch
    from eridiffusion_amd import _lib as L
    sizes = [2048 * 6 + 100, 640, 2048, 5120, 33]
    ps, gs = hs.make_inputs(sizes, bf16, 71 + bf16, g_std=1e-2)
    copies = []
    for _ in range(2):
        states = hs.oracle_states(sizes)
        gt = hs.GpuTensors([p.copy() for p in ps], [g.copy() for g in gs], states, bf16)
        rows = gt.rows()
        table = C.c_void_p()
        L.check(L.lib().eri_adam8_table_create(rows, len(rows), None, C.byref(table)), "table_create")
        copies.append((gt, table))
    (gt_e, tab_e), (gt_g, tab_g) = copies
    h = L.hyper_pack(LR, B1, B2, EPS, WD, 3, L.MODE_ERI, L.FLAG_CLIP_FROM_TABLE)

    def issue(table, stream):
        L.check(L.lib().eri_adam8_grad_norm(table, 0.05, 0.0, stream), "grad_norm")
        L.check(L.lib().eri_adam8_step_table(table, C.byref(h), stream), "step_table")

    # warm-up outside the capture: the first norm pass allocates the table's partial sums
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        issue(tab_g, side.cuda_stream)
    side.synchronize()
    issue(tab_e, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        issue(tab_g, torch.cuda.current_stream().cuda_stream)
    for replay in range(4):
        graph.replay()
        issue(tab_e, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        pe, se = gt_e.fetch()
        pg, sg = gt_g.fetch()
        for a, b in zip(pe, pg):
            assert np.array_equal(a, b), replay
        for sa, sb in zip(se, sg):
            for a, b in zip(sa, sb):
                assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), replay
        na, nb_ = C.c_float(), C.c_float()
        sc_a, sc_b = C.c_float(), C.c_float()
        L.check(L.lib().eri_adam8_grad_norm_read(tab_e, C.byref(na), C.byref(sc_a), None), "read")
        L.check(L.lib().eri_adam8_grad_norm_read(tab_g, C.byref(nb_), C.byref(sc_b), None), "read")
        assert na.value == nb_.value and sc_a.value == sc_b.value and sc_a.value < 1.0
        # eager work between replays: new gradients for both copies
        scratch = torch.randn(512, 512, device="cuda")
        scratch = (scratch @ scratch).sum()  # unrelated eager work, library reductions included
        fresh = hs.fresh_grads(sizes, bf16, 500 + replay, 1e-2)
        gt_e.set_grads(fresh)
        gt_g.set_grads(fresh)
        torch.cuda.synchronize()
    L.lib().eri_adam8_table_destroy(tab_e)
    L.lib().eri_adam8_table_destroy(tab_g)


def _tensors(sizes, seed):
    """Rows of bf16 tensors with shadows, and the memory they stand for."""
    import torch
    from eridiffusion_amd import _lib as L
    gen = torch.Generator(device="cuda").manual_seed(seed)
    blocks = [(n + 2047) // 2048 for n in sizes]
    total = sum(blocks)
    p, g, shadow = ((torch.randn(total * 2048, device="cuda", generator=gen) * s).to(torch.bfloat16) for s in (0.02, 1e-3, 0.01))
    m, v = (torch.empty(total * 2048, dtype=torch.uint8, device="cuda") for _ in range(2))
    am, av = (torch.empty(total, device="cuda") for _ in range(2))
    stream = torch.cuda.current_stream().cuda_stream
    L.check(L.lib().eri_adam8_state_init(m.data_ptr(), v.data_ptr(), am.data_ptr(), av.data_ptr(), m.numel(), stream), "state_init")
    m32, v32 = (torch.zeros(total * 2048, device="cuda") for _ in range(2))
    rows, rows32, ema, at = (L.TensorRow * len(sizes))(), (L.AdamW32Row * len(sizes))(), (L.EmaRow * len(sizes))(), 0
    for r, r32, e, n, b in zip(rows, rows32, ema, sizes, blocks):
        o = at * 2048
        r.p, r.g, r.ema_shadow = (x[o:].data_ptr() for x in (p, g, shadow))
        r.m, r.v, r.absmax_m, r.absmax_v = m[o:].data_ptr(), v[o:].data_ptr(), am[at:].data_ptr(), av[at:].data_ptr()
        r.numel, r.block_start, r.grad_scale, r.dtype_tag = n, at, 1.0, L.DTYPE_BF16
        r32.p, r32.g, r32.m, r32.v, r32.numel, r32.dtype_tag = r.p, r.g, m32[o:].data_ptr(), v32[o:].data_ptr(), n, L.DTYPE_BF16
        e.shadow, e.p, e.numel, e.dtype_tag = r.ema_shadow, r.p, n, L.DTYPE_BF16
        at += b
    table = C.c_void_p()
    L.check(L.lib().eri_adam8_table_create(rows, len(rows), stream, C.byref(table)), "table_create")
    return table, rows32, ema, (p, g, shadow, m, v, am, av, m32, v32)


@pytest.mark.parametrize("what", ["step", "sweeps"])
def test_graphs_of_launches_that_take_tickets(what):
    """More rounds than workgroups: a replay, an eager launch over the same rows and the next replay each find the counter
    where they need it."""
    import torch
    from eridiffusion_amd import _lib as L
    sizes = ([(64 * 256) * 2048 + 100, 3 * 2048, 5000] if what == "step" else [(128 * 256) * 2048 + 100, 3 * 2048, 5000])
    eager, graphed = _tensors(sizes, 7), _tensors(sizes, 7)
    hypers = []
    for flags in (0, L.FLAG_EMA):
        h = L.hyper_pack(LR, B1, B2, EPS, WD, 3, L.MODE_ERI, flags)
        h.ema_decay = 0.9
        hypers.append(h)
    h32 = L.AdamW32Hyper(LR, B1, B2, EPS, WD)

    def issue(tensors, stream):
        table, rows32, ema, _ = tensors
        if what == "step":
            for h in hypers:
                L.check(L.lib().eri_adam8_step_table(table, C.byref(h), stream), "step_table")
        else:
            L.check(L.lib().eri_adamw32_step_multi(rows32, len(rows32), C.byref(h32), stream), "adamw32")
            L.check(L.lib().eri_ema_update_multi(ema, len(ema), 0.9, stream), "ema")

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    issue(graphed, side.cuda_stream)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        issue(graphed, torch.cuda.current_stream().cuda_stream)
    main = torch.cuda.current_stream().cuda_stream
    issue(eager, main)
    for replay in range(4):
        graph.replay()
        issue(eager, main)
        issue(graphed, main)
        issue(eager, main)
        torch.cuda.synchronize()
        for a, b in zip(eager[3], graphed[3]):
            assert torch.equal(a, b), replay
    for tensors in (eager, graphed):
        L.lib().eri_adam8_table_destroy(tensors[0])
