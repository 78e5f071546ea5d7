"""Two host threads, two optimizers, two streams: the ABI is re-entrant on distinct handles
(the reference requires `Send + Sync` of an optimizer, crates/training/src/optimizer.rs:11)."""
import ctypes as C
import threading

import numpy as np
import pytest

import harness as hs

pytestmark = pytest.mark.gpu
LR, B1, B2, EPS, WD = 1e-4, 0.9, 0.999, 1e-8, 0.01


def _worker(idx, bf16, steps, out, barrier):
    import torch
    from eridiffusion_amd import _lib as L
    try:
        torch.cuda.set_device(0)
        sizes = [2048 * (9 + idx) + 13 * (idx + 1), 640 * 16, 2048, 77 + idx]
        ps, gs = hs.make_inputs(sizes, bf16, 400 + idx)
        states = hs.oracle_states(sizes)
        gt = hs.GpuTensors(ps, gs, states, bf16)
        stream = C.c_void_p()
        L.check(L.lib().eri_hip_stream_create(C.byref(stream)), "stream_create")
        torch.cuda.synchronize()  # the uploads above ran on torch's stream
        rows = gt.rows()
        table = C.c_void_p()
        # the table is uploaded on the NULL stream and stepped on the thread's own stream
        L.check(L.lib().eri_adam8_table_create(rows, len(rows), None, C.byref(table)), "table_create")
        barrier.wait()
        all_g = [gs] + [hs.fresh_grads(sizes, bf16, 9000 + 100 * idx + k) for k in range(1, steps)]
        for k in range(steps):
            if k:
                L.check(L.lib().eri_hip_stream_sync(stream), "sync")
                gt.set_grads(all_g[k])
                torch.cuda.synchronize()
            h = L.hyper_pack(LR, B1, B2, EPS, WD, k + 1, L.MODE_ERI, L.FLAG_EXACT_PARAM)
            L.check(L.lib().eri_adam8_grad_norm(table, 1e9, 0.0, stream), "grad_norm")
            L.check(L.lib().eri_adam8_step_table(table, C.byref(h), stream), "step_table")
            # a bad call on this thread leaves its message on this thread only
            assert L.lib().eri_adam8_step_table(None, C.byref(h), stream) == -1
            assert b"NULL" in L.lib().eri_last_error()
        L.check(L.lib().eri_hip_stream_sync(stream), "sync")
        for k in range(steps):
            hs.oracle_step(ps, all_g[k], states, (LR, B1, B2, EPS, WD, k + 1), bf16, threads=2)
        got_p, got_st = gt.fetch()
        stats = hs.compare(got_p, got_st, ps, states, bf16, True, "thread %d" % idx)
        assert stats["code_mismatch"] == 0
        L.lib().eri_adam8_table_destroy(table)
        L.lib().eri_hip_stream_destroy(stream)
        out[idx] = "ok"
    except BaseException as e:  # reported by the main thread
        out[idx] = repr(e)
        try:
            barrier.abort()
        except Exception:
            pass


@pytest.mark.parametrize("bf16", [True, False])
def test_two_threads_two_streams_each_bit_exact(bf16):
    out = {}
    barrier = threading.Barrier(2)
    threads = [threading.Thread(target=_worker, args=(i, bf16, 4, out, barrier)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert out == {0: "ok", 1: "ok"}, out


def test_step_multi_on_two_streams_of_one_thread():
    """The launch table behind eri_adam8_step_multi is not given other rows while a step that is queued on another
    stream has still to read it.  Both sets of rows against the same steps on one stream."""
    import torch
    from eridiffusion_amd import _lib as L
    sizes = [2048 * 5, 2048 + 9, 640]
    gen = torch.Generator(device="cuda").manual_seed(4)

    def make():
        one = []
        for n in sizes:
            nb = (n + 2047) // 2048
            t = [torch.randn(n, device="cuda", generator=gen), torch.randn(n, device="cuda", generator=gen),
                 torch.empty(n, dtype=torch.uint8, device="cuda"), torch.empty(n, dtype=torch.uint8, device="cuda"),
                 torch.empty(nb, device="cuda"), torch.empty(nb, device="cuda")]
            L.check(L.lib().eri_adam8_state_init(*[x.data_ptr() for x in t[2:]], n, None), "state_init")
            one.append(t)
        return one

    def step(one, t, stream):
        rows, start = (L.TensorRow * len(sizes))(), 0
        for r, n, x in zip(rows, sizes, one):
            r.p, r.g, r.m, r.v, r.absmax_m, r.absmax_v = [y.data_ptr() for y in x]
            r.numel, r.block_start, r.dtype_tag, r.grad_scale = n, start, L.DTYPE_F32, 1.0
            start += (n + 2047) // 2048
        h = L.hyper_pack(1e-3, 0.9, 0.999, 1e-8, 0.01, t, L.MODE_ERI, 0)
        L.check(L.lib().eri_adam8_step_multi(rows, len(rows), C.byref(h), stream.cuda_stream), "step_multi")
    sets = [make(), make()]
    torch.cuda.synchronize()
    want = [[[x.clone() for x in t] for t in one] for one in sets]
    a, b, default = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.current_stream()
    torch.cuda.synchronize()
    step(sets[0], 1, a)
    a.synchronize()
    with torch.cuda.stream(a):
        torch.cuda._sleep(5000000)
    step(sets[0], 2, a)
    step(sets[1], 1, b)
    step(sets[0], 3, a)
    step(sets[1], 2, b)
    torch.cuda.synchronize()
    for one, steps in zip(want, (3, 2)):
        for t in range(steps):
            step(one, t + 1, default)
    torch.cuda.synchronize()
    for got, expected in zip(sets, want):
        for x, y in zip(got, expected):
            assert all(torch.equal(u, v) for u, v in zip(x, y))
