"""Launches whose workgroups take their rounds of blocks by ticket: lists that end at, just before and just behind a
round, fewer rounds than workgroups and more, and the same table launched again and again (the counter is back at zero
each time), against the oracle, bit for bit."""
import ctypes as C

import pytest

import harness as hs

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
