"""Tables large enough for every route of the dispatch between the step kernels, and for a wave's second block: every
layout and mode against the prefetching kernel (which the parity tests hold against the oracle) on the same inputs, bit
for bit."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu
BLOCK = 2048


def _sizes(blocks, tail=0):
    """Elements of tensors with `blocks` full blocks in all; every other tensor has a partial block of about `tail`."""
    out, left = [], blocks
    while left > 0:
        n = min(1 + len(out) * 7 % 53, left)
        left -= n
        out.append(n * BLOCK + (tail + len(out) % 9 if tail and len(out) % 2 else 0))
    return out


def _run(layout, mode, sizes, flags, scale, ema=False):
    """Two steps over tensors of these sizes, some of them with a shadow if `ema`; returns everything the steps write."""
    import torch
    from eridiffusion_amd import _lib as L
    stream = torch.cuda.current_stream().cuda_stream
    blocks = sum((n + BLOCK - 1) // BLOCK for n in sizes)
    gen = torch.Generator(device="cuda").manual_seed(blocks + mode)
    pdt = torch.float32 if layout == "f32" else torch.bfloat16
    gdt = torch.bfloat16 if layout == "bf16" else torch.float32
    p = (torch.randn(blocks * BLOCK, device="cuda", generator=gen) * 0.02).to(pdt)
    gs = [(torch.randn(blocks * BLOCK, device="cuda", generator=gen) * 1e-3).to(gdt) for _ in range(2)]
    m, v = (torch.empty(blocks * BLOCK, dtype=torch.uint8, device="cuda") for _ in range(2))
    am, av = (torch.empty(blocks, device="cuda") for _ in range(2))
    shadow = p * 0.5
    L.check(L.lib().eri_adam8_state_init(m.data_ptr(), v.data_ptr(), am.data_ptr(), av.data_ptr(), m.numel(), stream), "init")
    for step, g in enumerate(gs, 1):
        rows, at = (L.TensorRow * len(sizes))(), 0
        for i, (r, n) in enumerate(zip(rows, sizes)):
            r.p, r.g = p.data_ptr() + at * BLOCK * p.element_size(), g.data_ptr() + at * BLOCK * g.element_size()
            r.m, r.v, r.absmax_m, r.absmax_v = m.data_ptr() + at * BLOCK, v.data_ptr() + at * BLOCK, am.data_ptr() + 4 * at, av.data_ptr() + 4 * at
            r.numel, r.block_start, r.grad_scale = n, at, 1.0
            r.dtype_tag, r.grad_f32 = (L.DTYPE_F32 if layout == "f32" else L.DTYPE_BF16), int(layout == "bf16-f32-grads")
            if ema and i % 3 != 1:
                r.ema_shadow = shadow.data_ptr() + at * BLOCK * p.element_size()
            at += (n + BLOCK - 1) // BLOCK
        h = L.hyper_pack(1e-3, 0.9, 0.999, 1e-8, 0.01, step - (mode == L.MODE_L2), mode, L.FLAG_EXACT_PARAM | flags | (L.FLAG_EMA if ema else 0), scale)
        h.ema_decay = 0.9
        L.check(L.lib().eri_adam8_step_multi(rows, len(rows), C.byref(h), stream), "step_multi")
    torch.cuda.synchronize()
    return p, m, v, am, av, shadow


@pytest.mark.parametrize("mode", [0, 1, 2], ids=["eri", "l2", "bnb"])
@pytest.mark.parametrize("layout", ["bf16", "bf16-f32-grads", "f32"])
@pytest.mark.parametrize("blocks,scale", [(1, None), (4097, 0.5), (96 * 256 + 300, None), (128 * 256 + 300, 0.5)])
def test_plain_kernel_over_whole_blocks(layout, mode, blocks, scale):
    """Without the code for partial blocks, on tables of its own size and of the prefetching kernel's."""
    import torch
    from eridiffusion_amd import _lib as L
    want = _run(layout, mode, _sizes(blocks), L.FLAG_ONE_WAVE, scale)
    got = _run(layout, mode, _sizes(blocks), L.FLAG_NO_PIPELINE, scale)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("mode", [0, 1, 2], ids=["eri", "l2", "bnb"])
@pytest.mark.parametrize("tail", [0, 515])
def test_split_kernel_over_several_rounds(mode, tail):
    """Its teams go round more than once only for fp32 gradients of bf16 parameters under the binary-search flag, at any
    table size: other tables of more than one round take the kernels with a wave per block."""
    import torch
    from eridiffusion_amd import _lib as L
    sizes = _sizes(3000, tail)
    want = _run("bf16-f32-grads", mode, sizes, L.FLAG_ONE_WAVE, 0.5)
    for a, b in zip(_run("bf16-f32-grads", mode, sizes, L.FLAG_BSEARCH, 0.5), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("layout,mode", [("bf16", 0), ("bf16-f32-grads", 0), ("f32", 0), ("bf16", 2), ("f32", 2)])
@pytest.mark.parametrize("blocks", [1024, 1025, 12 * 256, 12 * 256 + 1, 64 * 256, 64 * 256 + 1])
@pytest.mark.parametrize("tail", [0, 515])
def test_every_route_of_a_step_with_an_ema(layout, mode, blocks, tail):
    """On both sides of each line between the kernels that take such a step."""
    import torch
    from eridiffusion_amd import _lib as L
    sizes = _sizes(blocks, tail)
    want = _run(layout, mode, sizes, L.FLAG_ONE_WAVE, None, ema=True)
    assert not torch.equal(want[5], _run(layout, mode, sizes, 0, None)[5])
    for a, b in zip(_run(layout, mode, sizes, 0, None, ema=True), want):
        assert torch.equal(a, b)
