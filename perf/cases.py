"""What a user of the library has it do, as cases that can be timed and compared.

A case is a dict of plain values.  `path` names the public entry points a pass goes through:

  list        Adam8bit.step() over torch tensors that carry `.grad` (the list optimizer)
  functional  update_params_8bit() over named tensors, then step() (the per-name optimizer)
  many        the per-name optimizer from C: eri_adam8bit_fn_update_many, each step into the other output set
  table       eri_adam8_step_table on a launch table, the gradient norm before it when the case clips
  checkpoint  load_state_from_tensors() of a saved set of fp32 moments, then get_state_as_tensors()
  adamw32     eri_adamw32_step_multi, the step for tensors kept in 32-bit moments

`shapes` names the tensor list (eridiffusion_amd/workloads.py, or generic ones built here), `take` a prefix of it.
Every state starts with the history of two steps on other gradients, as a training run has it.
"""
import ctypes as C
import math
import random

import torch

from eridiffusion_amd import _lib as L
from eridiffusion_amd import workloads as W
from eridiffusion_amd.adam8bit import Adam8bit, Adam8bitConfig, Adam8bitFunctional, DevicePool, update_params_8bit

HYPER = (1e-4, 0.9, 0.999, 1e-8, 0.01)  # lr, beta1, beta2, eps, weight decay
EMA_DECAY = 0.9999
CHUNK = 1 << 30  # elements of one output; larger arrays come back as several views


def _case(**given):
    """Every case says all of its choices."""
    case = dict(path="list", shapes="flat", rank=0, pairs=0, elems=0, count=0, take=0, dtype="bf16", grad="same", clip=False,
                min8=0, ema=False, exact=True, fresh=False, master=False)
    case.update(given)
    return case


def listed():
    return [
        # one flat fp32 tensor of a million parameters: the smallest step, where launch and latency count
        _case(name="flat_1m_f32", path="list", shapes="flat", elems=1 << 20, dtype="f32"),
        # a rank-16 adapter on the first blocks of a transformer, named tensors, fp32 gradients straight from autograd
        _case(name="flux_lora_first_blocks", path="functional", shapes="flux_lora", rank=16, take=60, grad="f32"),
        # a small adapter under the trainers' usual settings: clipping, short tensors in 32 bits, gradients at new
        # addresses every step
        _case(name="sdxl_lora_r4_trainer", path="list", shapes="sdxl_lora", rank=4, pairs=128, clip=True, min8=4096, fresh=True),
        # norms, biases, embeddings and odd widths, both parameter dtypes in one optimizer
        _case(name="ragged_mixed", path="list", shapes="ragged", count=400, elems=300001, dtype="mixed"),
        # the rank-16 adapter on all of an SDXL-sized UNet, through the list optimizer
        _case(name="sdxl_lora_r16", path="list", shapes="sdxl_lora", rank=16, pairs=700),
        # the same adapter through the per-name optimizer
        _case(name="sdxl_lora_r16_named", path="many", shapes="sdxl_lora", rank=16, pairs=700),
        # the rank-32 adapter on every linear of a FLUX-sized transformer, gradients clipped by their global norm
        _case(name="flux_lora_r32_clip", path="table", shapes="flux_lora", rank=32, clip=True),
        # the moments of one transformer block out of a checkpoint and into the next one
        _case(name="checkpoint_block", path="checkpoint", shapes="flux_block"),
        # full fine-tune of an SDXL-sized UNet with the EMA of the weights, fp32 gradients, clipped
        _case(name="sdxl_full_ema", path="table", shapes="sdxl_full", grad="f32", ema=True, clip=True),
        # full fine-tune of an SDXL-sized UNet held in fp32
        _case(name="sdxl_full_f32", path="table", shapes="sdxl_full", dtype="f32"),
        # half of that UNet with 32-bit moments
        _case(name="sdxl_half_adamw32", path="adamw32", shapes="sdxl_full", take=840),
        # full fine-tune of a FLUX-12B-sized model with the faster parameter arithmetic
        _case(name="flux_full", path="table", shapes="flux_full", exact=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    path = rng.choice(["list", "list", "functional", "many", "table", "table", "table", "checkpoint", "adamw32"])
    case = _case(path=path)
    # the kind of tensor list the path is used on
    small = ["flat", "sdxl_lora", "flux_lora", "ragged"]
    kind = {"list": small, "functional": ["flux_lora", "flux_block"], "many": ["sdxl_lora", "flux_lora"],
            "table": small + ["sdxl_full", "sdxl_full", "flux_full"], "checkpoint": ["flux_block", "flux_lora"],
            "adamw32": ["ragged", "sdxl_full"]}[path]
    shapes = case["shapes"] = rng.choice(kind)
    named = path in ("functional", "checkpoint")  # these return every tensor on its own: not more than a block's worth
    if shapes == "flat":
        case["elems"] = _log_int(rng, 1 << 12, 1 << 26)
    elif shapes == "ragged":
        case["count"], case["elems"] = _log_int(rng, 10, 1000), _log_int(rng, 1000, 1000000)
    elif shapes == "sdxl_lora":
        case["rank"], case["pairs"] = _log_int(rng, 2, 64), _log_int(rng, 10, 700)
    elif shapes == "flux_lora":
        case["rank"], case["take"] = _log_int(rng, 2, 128), rng.randint(8, 30) if named else _log_int(rng, 20, 608)
    elif shapes == "flux_block":
        case["take"] = rng.randint(3, 24)
    elif shapes == "sdxl_full":
        case["take"] = _log_int(rng, 50, 1680)
    elif shapes == "flux_full":
        case["take"] = _log_int(rng, 16, 400)
    if path == "list":
        case["dtype"] = "mixed" if shapes == "ragged" else rng.choice(["bf16", "bf16", "f32"])
        case["clip"], case["min8"], case["fresh"] = rng.random() < 0.5, rng.choice([0, 0, 4096]), rng.random() < 0.3
    elif path == "table":
        case["dtype"] = "mixed" if shapes == "ragged" else rng.choice(["bf16", "bf16", "f32"])
        case["grad"] = rng.choice(["same", "same", "f32"]) if case["dtype"] == "bf16" else "same"
        case["clip"], case["ema"], case["exact"] = rng.random() < 0.3, rng.random() < 0.25, rng.random() < 0.6
    elif path == "functional":
        case["grad"] = rng.choice(["same", "f32"])
    elif path == "adamw32":
        case["dtype"], case["master"] = rng.choice(["bf16", "f32"]), False
        case["master"] = case["dtype"] == "bf16" and rng.random() < 0.5
    return case


# ---------------------------------------------------------------------------------------------------------------
# tensor lists
# ---------------------------------------------------------------------------------------------------------------

def _tensors(case):
    """[(name, shape, dtype)] of the case, dtype being "bf16" or "f32"."""
    kind = case["shapes"]
    if kind == "flat":
        out = [("flat", (case["elems"],))]
    elif kind == "ragged":  # sizes spread over their logarithm, most of them odd
        r = random.Random(case["count"] * 1000003 + case["elems"])
        out = [("t.%d" % i, (_log_int(r, 1, case["elems"]),)) for i in range(case["count"])]
    elif kind == "sdxl_lora":
        out = W.c2_sdxl_lora(rank=case["rank"], pairs=case["pairs"])
    elif kind == "flux_lora":
        out = W.c3_flux_lora(rank=case["rank"])
    elif kind == "flux_block":
        out = [t for t in W.c5_flux_full() if t[0].startswith("double_blocks.0.")]
    elif kind == "sdxl_full":
        out = W.c4_sdxl_full()
    else:
        out = W.c5_flux_full()
    if case["take"]:
        out = out[:case["take"]]
    mixed = case["dtype"] == "mixed"
    return [(n, s, ("f32" if i % 4 == 3 else "bf16") if mixed else case["dtype"]) for i, (n, s) in enumerate(out)]


def _std(case, name, shape):
    config = {"sdxl_lora": "c2_sdxl_lora_r16", "flux_lora": "c3_flux_lora_r32"}.get(case["shapes"], "")
    return W.init_std(config, name, shape)


def _blocks(n):
    return (n + L.BLOCK - 1) // L.BLOCK


def _align(n):
    return (n + 255) // 256 * 256


DT = {"bf16": torch.bfloat16, "f32": torch.float32}
TAG = {"bf16": L.DTYPE_BF16, "f32": L.DTYPE_F32}
SIZE = {"bf16": 2, "f32": 4}


class Arena:
    """One device array that holds a list of tensors, each on a 256-byte boundary."""

    def __init__(self, dtypes, sizes):
        self.offsets, total = [], 0
        for n, dt in zip(sizes, dtypes):
            self.offsets.append(total)
            total += _align(n * torch.empty(0, dtype=dt).element_size())
        self.raw = torch.zeros(total, dtype=torch.uint8, device="cuda")
        self.dtypes, self.sizes = dtypes, sizes
        self.base = self.raw.data_ptr()

    def ptr(self, i):
        return self.base + self.offsets[i]

    def view(self, i):
        dt = self.dtypes[i]
        size = torch.empty(0, dtype=dt).element_size()
        return self.raw[self.offsets[i]:self.offsets[i] + self.sizes[i] * size].view(dt)

    def whole(self):
        """The array as it stands, by its tensors' common dtype (bytes if they have several)."""
        flat = self.raw.view(self.dtypes[0]) if len(set(self.dtypes)) == 1 else self.raw
        return list(flat.split(CHUNK))

    def normal(self, stds, gen):
        """Fills every tensor with normal values of its own spread."""
        if len(set(stds)) == 1 and len(set(self.dtypes)) == 1:
            for part in self.raw.view(self.dtypes[0]).split(CHUNK):
                part.normal_(0.0, stds[0], generator=gen)
        else:
            for i, std in enumerate(stds):
                self.view(i).normal_(0.0, std, generator=gen)


class _Pooled:
    """The bytes a lane of a pool has handed out, as torch sees foreign device memory; holds the pool."""

    def __init__(self, pool, ptr, nbytes):
        self.pool = pool
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (ptr, False), "version": 2}


class StatePool:
    """A pool of one lane that an optimizer takes its 8-bit states from, so that they can be looked at whole."""

    def __init__(self, sizes):
        need = 256 + sum(2 * _align(n) + 2 * _align(4 * _blocks(n)) for n in sizes)
        self.pool = DevicePool((need + (2 << 20) - 1) // (2 << 20) * (2 << 20), 1)
        self.base = self.pool.alloc_ptr(0, 256)

    def states(self):
        used = C.c_size_t()
        L.check(L.lib().eri_hip_pool_lane_used(self.pool._pool, 0, C.byref(used)), "eri_hip_pool_lane_used")
        out = torch.as_tensor(_Pooled(self.pool, self.base, used.value), device="cuda")
        out.pool = self.pool  # the pool's memory lives as long as what is returned, also past the optimizer
        return out


class State:
    """What the user's program keeps between passes."""
    table = named = None

    def __del__(self):
        if self.table:
            L.lib().eri_adam8_table_destroy(self.table)
        if self.named:
            L.lib().eri_adam8bit_fn_destroy(self.named)


def _stream():
    return torch.cuda.current_stream().cuda_stream


# ---------------------------------------------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    s = State()
    s.case, s.t = case, 0
    s.gen = torch.Generator(device="cuda")
    s.gen.manual_seed(seed)
    s.tensors = _tensors(case)
    s.sizes = [W.numel(shape) for _, shape, _ in s.tensors]
    stds = [_std(case, name, shape) for name, shape, _ in s.tensors]
    s.p_std, s.g_std = [a for a, _ in stds], [b for _, b in stds]
    return {"list": _prepare_list, "functional": _prepare_functional, "many": _prepare_many, "table": _prepare_table,
            "checkpoint": _prepare_checkpoint, "adamw32": _prepare_adamw32}[case["path"]](s)


def _params(s):
    dts = [DT[d] for _, _, d in s.tensors]
    s.p = Arena(dts, s.sizes)
    s.p.normal(s.p_std, s.gen)
    gdts = [torch.float32] * len(dts) if s.case["grad"] == "f32" else dts
    s.g = Arena(gdts, s.sizes)
    s.g.normal(s.g_std, s.gen)
    return dts, gdts


def _history(s, grads=None):
    """Two passes on other gradients; the gradients of the passes to come are new ones."""
    for _ in range(2):
        run(s)
        for g in grads or [s.g]:
            g.normal(s.g_std, s.gen)


def _prepare_list(s):
    _, gdts = _params(s)
    params = [s.p.view(i).view(shape) for i, (_, shape, _) in enumerate(s.tensors)]
    arenas = [s.g]
    if s.case["fresh"]:
        arenas.append(Arena(gdts, s.sizes))
        arenas[1].normal(s.g_std, s.gen)
    s.grads = [[a.view(i).view(shape) for i, (_, shape, _) in enumerate(s.tensors)] for a in arenas]
    s.params = params
    for p, g in zip(params, s.grads[0]):
        p.grad = g
    lr, b1, b2, eps, wd = HYPER
    s.opt = Adam8bit(params, Adam8bitConfig(lr=lr, betas=(b1, b2), eps=eps, weight_decay=wd, min_8bit_size=s.case["min8"]))
    s.pool = StatePool(s.sizes)
    s.opt.set_state_pool(s.pool.pool, 0)
    if s.case["clip"]:
        s.opt.set_max_grad_norm(1e-1)
    _history(s, arenas)
    return s


def _prepare_functional(s):
    _params(s)
    names = [n for n, _, _ in s.tensors]
    s.params = {n: s.p.view(i).view(s.tensors[i][1]) for i, n in enumerate(names)}
    s.grads = {n: s.g.view(i).view(s.tensors[i][1]) for i, n in enumerate(names)}
    s.opt = Adam8bitFunctional.with_params(*HYPER)
    s.pool = StatePool(s.sizes)
    s.opt.set_state_pool(s.pool.pool, 0)
    _history(s)
    return s


def _prepare_many(s):
    dts, _ = _params(s)
    s.p2 = Arena(dts, s.sizes)
    n = len(s.sizes)
    s.named = C.c_void_p()
    L.check(L.lib().eri_adam8bit_fn_with_params(*HYPER, _stream(), C.byref(s.named)), "fn_with_params")
    s.pool = StatePool(s.sizes)
    L.check(L.lib().eri_adam8bit_fn_set_state_pool(s.named, s.pool.pool._pool, 0), "fn_set_state_pool")
    s.names = (C.c_char_p * n)(*[name.encode() for name, _, _ in s.tensors])
    s.numels = (C.c_uint64 * n)(*s.sizes)
    s.tags = (C.c_int32 * n)(*[TAG[d] for _, _, d in s.tensors])

    def ptrs(a):
        return (C.c_void_p * n)(*[a.ptr(i) for i in range(n)])
    s.c_g = ptrs(s.g)
    s.sets = [(ptrs(s.p), ptrs(s.p2), s.p2), (ptrs(s.p2), ptrs(s.p), s.p)]
    _history(s)
    return s


def _prepare_table(s):
    dts, gdts = _params(s)
    u8, f32 = [torch.uint8] * len(dts), [torch.float32] * len(dts)
    nb = [_blocks(n) for n in s.sizes]
    s.m, s.v, s.am, s.av = Arena(u8, s.sizes), Arena(u8, s.sizes), Arena(f32, nb), Arena(f32, nb)
    for i, n in enumerate(s.sizes):
        L.check(L.lib().eri_adam8_state_init(s.m.ptr(i), s.v.ptr(i), s.am.ptr(i), s.av.ptr(i), n, _stream()), "state_init")
    s.shadow = None
    if s.case["ema"]:
        s.shadow = Arena(dts, s.sizes)
        s.shadow.raw.copy_(s.p.raw)
    s.rows = (L.TensorRow * len(dts))()
    start = 0
    for i, n in enumerate(s.sizes):
        r = s.rows[i]
        r.p, r.g, r.m, r.v, r.absmax_m, r.absmax_v = s.p.ptr(i), s.g.ptr(i), s.m.ptr(i), s.v.ptr(i), s.am.ptr(i), s.av.ptr(i)
        r.numel, r.block_start, r.dtype_tag, r.grad_scale = n, start, TAG[s.tensors[i][2]], 1.0
        r.grad_f32 = 1 if dts[i] == torch.bfloat16 and gdts[i] == torch.float32 else 0
        if s.shadow is not None:
            r.ema_shadow = s.shadow.ptr(i)
        start += nb[i]
    s.table = C.c_void_p()
    L.check(L.lib().eri_adam8_table_create(s.rows, len(s.rows), _stream(), C.byref(s.table)), "table_create")
    _history(s)
    return s


def _prepare_checkpoint(s):
    f32 = [torch.float32] * len(s.sizes)
    s.m, s.v = Arena(f32, s.sizes), Arena(f32, s.sizes)
    s.m.normal([g * 0.3 for g in s.g_std], s.gen)
    s.v.normal(s.g_std, s.gen)
    s.v.raw.view(torch.float32).square_()
    s.saved = {name: (s.m.view(i), s.v.view(i)) for i, (name, _, _) in enumerate(s.tensors)}
    s.opt = Adam8bitFunctional.with_params(*HYPER)
    run(s)  # an optimizer that already has states
    return s


def _prepare_adamw32(s):
    dts, _ = _params(s)
    f32 = [torch.float32] * len(dts)
    s.m, s.v = Arena(f32, s.sizes), Arena(f32, s.sizes)
    s.w = None
    if s.case["master"]:
        s.w = Arena(f32, s.sizes)
        for i in range(len(dts)):
            s.w.view(i).copy_(s.p.view(i))
    s.rows = (L.AdamW32Row * len(dts))()
    for i, n in enumerate(s.sizes):
        r = s.rows[i]
        r.p, r.g, r.m, r.v, r.numel, r.dtype_tag = s.p.ptr(i), s.g.ptr(i), s.m.ptr(i), s.v.ptr(i), n, TAG[s.tensors[i][2]]
        if s.w is not None:
            r.master = s.w.ptr(i)
    s.hyper = L.AdamW32Hyper(*HYPER)
    _history(s)
    return s


# ---------------------------------------------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------------------------------------------

def run(s):
    s.t += 1
    return {"list": _run_list, "functional": _run_functional, "many": _run_many, "table": _run_table,
            "checkpoint": _run_checkpoint, "adamw32": _run_adamw32}[s.case["path"]](s)


def _run_list(s):
    if len(s.grads) > 1:  # a backward pass left its gradients in other memory than the one before
        for p, g in zip(s.params, s.grads[s.t & 1]):
            p.grad = g
    s.opt.step()
    return [s.p.whole(), s.pool.states()]


def _run_functional(s):
    update_params_8bit(s.opt, s.params, s.grads)
    s.opt.step()
    return [list(s.params.values()), s.pool.states()]


def _run_many(s):
    src, dst, out = s.sets[s.t & 1]
    L.check(L.lib().eri_adam8bit_fn_update_many(s.named, s.names, src, s.c_g, s.numels, s.tags, None, dst, len(s.sizes)),
            "fn_update_many")
    L.check(L.lib().eri_adam8bit_fn_step(s.named), "fn_step")
    return [out.whole(), s.pool.states()]


def _run_table(s):
    case, stream = s.case, _stream()
    flags = L.FLAG_EXACT_PARAM if case["exact"] else 0
    if case["clip"]:
        L.check(L.lib().eri_adam8_grad_norm(s.table, 1e-1, 0.0, stream), "grad_norm")
        flags |= L.FLAG_CLIP_FROM_TABLE
    if case["ema"]:
        flags |= L.FLAG_EMA
    h = L.hyper_pack(*HYPER, s.t, L.MODE_ERI, flags)
    h.ema_decay = EMA_DECAY
    L.check(L.lib().eri_adam8_step_table(s.table, C.byref(h), stream), "step_table")
    arrays = [s.p, s.m, s.v, s.am, s.av] + ([s.shadow] if s.shadow is not None else [])
    return [a.whole() for a in arrays]


def _run_checkpoint(s):
    s.opt.load_state_from_tensors(s.saved)
    return s.opt.get_state_as_tensors()


def _run_adamw32(s):
    L.check(L.lib().eri_adamw32_step_multi(s.rows, len(s.rows), C.byref(s.hyper), _stream()), "adamw32")
    return [a.whole() for a in [s.p, s.m, s.v] + ([s.w] if s.w is not None else [])]


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two correct answers may be apart
# ---------------------------------------------------------------------------------------------------------------

def work(case):
    read_write = flops = 0.0
    for name, shape, dt in _tensors(case):
        n = W.numel(shape)
        p, g = SIZE[dt], 4 if case["grad"] == "f32" else SIZE[dt]
        if case["path"] == "checkpoint":  # fp32 moments in, states written, fp32 moments out
            read_write += n * (8 + 2 + 8) + 8 * _blocks(n)
            flops += n * 8
        elif case["path"] == "adamw32" or (case["min8"] and n < case["min8"]):
            read_write += n * (g + 16 + (p + 8 if case["master"] else 2 * p))
            flops += n * 14
        else:
            read_write += n * (2 * p + g + 4 + (2 * p if case["ema"] else 0)) + 16 * _blocks(n)
            flops += n * (20 + (3 if case["ema"] else 0) + (2 if case["clip"] else 0))
    return {"bytes": read_write, "flops": flops}


def tolerance(case):
    """States and exact parameters are specified bit for bit.  The faster parameter arithmetic may differ by one
    bf16 step of the parameter (2^-7 of it) in about one element of a million (2e-6 of the whole seen).  The clip
    factor may differ in its last bit with the order of the sums behind it; moments then differ by a few 2^-24, which
    moves absmax (2e-5 of the whole and 5e-3 of single ones seen after three steps), its bytes and those codes and
    bf16 roundings that lie on an edge (1e-4 of the state's bytes, absmax among them)."""
    if case["path"] in ("checkpoint", "adamw32"):
        return "exact"
    if case["clip"]:
        return {"rel": 1e-4, "max": 0.02, "differ": 5e-4}
    if not case["exact"] and case["dtype"] != "f32":
        return {"rel": 1e-5, "max": 0.008, "differ": 0.0}
    return "exact"
