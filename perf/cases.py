"""What is timed: the framework's work through its public entry points.

Two kinds of case:

* ``row`` - one pipeline rank's row of a schedule's task table on a ``StageExecutor``, driven by
  ``RankLoop``: every forward and backward task of the rank, gradients accumulated in fp32 from
  zero, boundary activations and cotangents in device buffers as they come from and go to the
  neighbouring ranks; optionally the Adam update behind the loop, optionally as a replay of a
  recorded HIP graph.
* ``step`` - a whole train step as a user writes it: ``mpmd_jit_with_loop`` around
  ``value_and_grad`` + ``treduce`` over all stages, then ``optim.adam`` and
  ``optim.apply_updates``, with the parameters, the optimizer state and the batch in host arrays.
"""
from __future__ import annotations

import math
from functools import partial

import numpy as np
import torch

import jaxpp_amd as jaxpp
from jaxpp_amd import runtime as rt
from jaxpp_amd import schedules as S
from jaxpp_amd.model import LayerSpec
from jaxpp_amd.plan import make_rank_plan
from jaxpp_amd.rank_loop import RankLoop
from jaxpp_amd.types import TaskType

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _case(name, kind, family, hidden, heads, ffn, seq, batch, layers, schedule, stages, n,
          kv=0, mpmd=0, rank=0, group=0, dtype="bf16", causal=None, tanh=False, adam=False,
          graph=False):
    """A case as a dict of plain values.  `layers` per stage; `mpmd` ranks of an interleaved
    schedule (0: one stage per rank); `n` microbatches; `group` microbatches whose weight
    gradients run as one product (0: each by itself)."""
    c = dict(kind=kind, family=family, hidden=hidden, heads=heads, kv=kv or heads, ffn=ffn, seq=seq,
             batch=batch, layers=layers, schedule=schedule, stages=stages, mpmd=mpmd, n=n, rank=rank,
             group=group, dtype=dtype, causal=family != "bert" if causal is None else causal,
             tanh=tanh, adam=adam, graph=graph)
    return {"name": name, **c} if name else c


def listed():
    return [
        # The smallest work the executor is given: one layer of hidden 128 on 128 tokens, two
        # microbatches.  A few dozen launches of a few microseconds; their number and latency
        # are everything.
        _case("smallest row", "row", "bert", 128, 2, 256, 128, 1, 1, "Std1F1B", 2, 2, rank=1),
        # examples/basic.py as it stands: four pre-LN decoder blocks of hidden 256 in two stages,
        # four microbatches, Adam; everything from and to host arrays.
        _case("example train step", "step", "decoder", 256, 2, 768, 128, 2, 2, "Std1F1B", 2, 4,
              tanh=True),
        # The float32 configuration (the reference's CPU-runnable one): four post-LN layers of
        # hidden 256 in two stages, eight microbatches of 4 x 128 tokens, the README's train step
        # with Adam.
        _case("float32 train step", "step", "bert", 256, 4, 1024, 128, 4, 2, "Std1F1B", 2, 8,
              dtype="f32"),
        # The same configuration's first rank alone, on device buffers.
        _case("float32 row", "row", "bert", 256, 4, 1024, 128, 4, 2, "Std1F1B", 2, 8, dtype="f32"),
        # An encoder of ordinary width whose sizes are multiples of 128 and of nothing larger:
        # 1152 tokens, hidden 768, sequences of 384.
        _case("odd encoder row", "row", "bert", 768, 12, 3072, 384, 3, 3, "Eager1F1B", 4, 6, rank=2),
        # Decoder blocks of hidden 1024 on 512 tokens a microbatch, two chunks per rank: the
        # middle of the range, where a product has fewer tiles than the device has CUs.
        _case("decoder row", "row", "decoder", 1024, 8, 4096, 256, 2, 2, "Interleaved1F1B", 4, 8,
              mpmd=2, tanh=True),
        # A rank's train step on a Llama-shaped stage of hidden 2048 (grouped-query heads, an odd
        # feed-forward width) with the ZeroBubble split and Adam over its parameters.
        _case("llama train row", "row", "llama", 2048, 16, 5632, 512, 1, 4, "ZeroBubble", 4, 8, kv=4,
              rank=1, adam=True),
        # The BERT-large-shaped benchmark workload: six layers, 16 microbatches of 8 x 512
        # tokens, recorded once and replayed, as the benchmark runs it.
        _case("bert-large graph row", "row", "bert", 1024, 16, 4096, 512, 8, 6, "Std1F1B", 4, 16,
              group=4, graph=True),
        # The headline workload's layer (Llama-3-8B-shaped, 4096 tokens a microbatch) and
        # schedule, one layer per chunk and eight microbatches.
        _case("llama-8b row", "row", "llama", 4096, 32, 14336, 4096, 1, 1, "Interleaved1F1B", 8, 8,
              kv=8, mpmd=4, group=4),
        # The 70B-shaped benchmark layer under ZeroBubble, one layer and four microbatches.
        _case("llama-70b row", "row", "llama", 8192, 64, 28672, 4096, 1, 1, "ZeroBubble", 4, 4, kv=8,
              rank=1, group=2),
        # The mixture-of-experts benchmark layer (top-2 of 8 experts, 2 x 4096 tokens) under
        # DualPipeV, one layer per chunk.  The largest.
        _case("mixtral row", "row", "mixtral", 4096, 32, 14336, 4096, 2, 1, "DualPipeV", 4, 4, kv=8,
              mpmd=2, group=2),
    ]


def _log_int(rng, lo, hi, unit):
    """A multiple of `unit` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / unit)) * unit))


def draw(rng):
    while True:
        kind = "step" if rng.random() < 0.2 else "row"
        family = rng.choice(["bert", "bert", "decoder", "decoder", "llama", "llama", "llama", "mixtral"])
        if kind == "step" and family == "mixtral":
            continue
        dtype = "f32" if rng.random() < (0.4 if kind == "step" else 0.2) else "bf16"
        small = kind == "step" or dtype == "f32"
        unit = 256 if family == "mixtral" else 128
        hidden = _log_int(rng, unit, 512 if small else 4096 if family in ("bert", "mixtral") else 8192, unit)
        head_dim = rng.choice([64, 128])
        heads = hidden // head_dim
        kv = rng.choice([k for k in (1, 2, 4, 8, heads) if k <= heads and heads % k == 0]) \
            if family in ("llama", "mixtral") else heads
        ffn = max(unit, int(round(hidden * rng.choice([2, 2.6875, 2.75, 3, 3.5, 4]) / unit)) * unit)
        seq = _log_int(rng, 128, 512 if small else 4096, 128)
        tokens = _log_int(rng, 128, 1024 if small else 8192, 128)
        batch = max(1, tokens // seq)
        layers = rng.randint(1, 2) if kind == "step" else rng.randint(1, 6)
        schedule = rng.choice(["Std1F1B", "Eager1F1B", "Interleaved1F1B", "ZeroBubble", "DualPipeV"])
        if schedule in ("Interleaved1F1B", "DualPipeV"):
            mpmd = 1 if kind == "step" else 2
            stages = 2 * mpmd
            n = mpmd * rng.randint(2, 5)
        else:
            mpmd, stages = 0, 2 if kind == "step" else rng.randint(2, 4)
            n = rng.randint(stages, 12)
        rank = 0 if kind == "step" else rng.randrange(mpmd or stages)
        group = rng.choice([0, 2, 4]) if not small and family != "decoder" and hidden >= 1024 else 0
        c = _case(None, kind, family, hidden, heads, ffn, seq, batch, layers, schedule, stages, n, kv=kv,
                  mpmd=mpmd, rank=rank, group=group, dtype=dtype,
                  causal=family in ("llama", "mixtral") or (family == "decoder" and rng.random() < 0.8),
                  tanh=family == "decoder" or rng.random() < 0.3,
                  adam=kind == "row" and rng.random() < 0.25, graph=kind == "row" and not small and
                  hidden < 2048 and rng.random() < 0.3)
        flops = work(c)["flops"]
        if flops > (1e11 if small else 1e14) or _device_bytes(c) > 40e9:
            continue
        if c["graph"] and c["adam"]:
            continue                # an update's step number is a launch argument: not recorded
        return c


# ---------------------------------------------------------------------------
def _spec(c) -> LayerSpec:
    moe = dict(n_experts=8, top_k=2) if c["family"] == "mixtral" else {}
    eps = 1e-12 if c["family"] == "bert" else 1e-6 if c["family"] == "decoder" else 1e-5
    return LayerSpec(c["family"], c["hidden"], c["heads"], c["ffn"], c["seq"], c["batch"],
                     n_kv_heads=c["kv"], causal=c["causal"], eps=eps, gelu_tanh=c["tanh"],
                     dtype=c["dtype"], **moe)


def _schedule(c):
    kw = {"num_stages": c["stages"]}
    if c["mpmd"]:
        kw["mpmd_dim"] = c["mpmd"]
    return getattr(S, c["schedule"])(**kw)


def _layer_elems(spec) -> int:
    return sum(int(np.prod(s)) for s in spec.param_shapes().values())


def _device_bytes(c) -> float:
    """Roughly what a case's state holds on the device."""
    spec = _spec(c)
    es = 4 if c["dtype"] == "f32" else 2
    if c["kind"] == "step":
        return _layer_elems(spec) * c["layers"] * c["stages"] * (es + 4)
    plan = make_rank_plan(_schedule(c), c["n"], c["rank"])
    T = spec.tokens * (3 if c["family"] == "mixtral" else 1)
    slot = c["layers"] * es * (spec.tokens * (8 * spec.hidden + 2 * spec.qkv_width) +
                               T * (2 * spec.hidden + 6 * spec.ffn))
    slots = plan.max_live + plan.n_chunks * max(0, c["group"] - 1)
    params = _layer_elems(spec) * c["layers"] * plan.n_chunks
    return params * (es + 4 + (12 if c["adam"] else 0)) + slots * slot + \
        4 * es * spec.tokens * spec.hidden * c["n"] * plan.n_chunks


def work(c):
    spec = _spec(c)
    es = 4 if c["dtype"] == "f32" else 2
    act = spec.tokens * spec.hidden
    if c["kind"] == "step":
        n_layers = c["layers"] * c["stages"]
        params = _layer_elems(spec) * n_layers
        # parameters, moments and the batch in; parameters, moments and predictions out
        nbytes = 4.0 * (6 * params + 2 * act * c["n"])
    else:
        chunks = make_rank_plan(_schedule(c), c["n"], c["rank"]).n_chunks
        n_layers = c["layers"] * chunks
        params = _layer_elems(spec) * n_layers
        # boundary tensors in and out, parameters in, gradients (or the updated state) out
        nbytes = 4.0 * es * act * c["n"] * chunks + params * (es + 4.0)
        if c["adam"]:
            nbytes += params * (24.0 + es)
    return {"bytes": nbytes, "flops": 3.0 * spec.fwd_flops() * n_layers * c["n"]}


def tolerance(c):
    """About four times what the outputs move by when hidden and feed-forward features are
    permuted - the same sums in another order: in float32 9e-7 (largest difference 1.1e-5), in
    bf16 on encoder and decoder stages 4e-3 (0.06; three layers), on Llama-shaped ones 9.6e-3
    (0.08; four layers, a stage in bf16 is 1e-2 from the same stage in float32); a mixture's
    token whose two best experts tie within rounding changes as a whole.  An Adam row's first
    updates are the sign of the gradient: of one that is zero within rounding, either sign
    (three passes of 1e-5 each way on a weight of 0.02)."""
    if c["dtype"] == "f32" and c["adam"]:
        return {"rel": 8e-6, "max": 5e-3}
    if c["dtype"] == "f32":
        return {"rel": 4e-6, "max": 5e-5}
    if c["family"] == "mixtral":
        return {"rel": 3e-2, "max": 1 - 1e-9}
    return {"rel": 3e-2, "max": 0.4} if c["family"] == "llama" else {"rel": 1.6e-2, "max": 0.25}


# ---------------------------------------------------------------------------
class _Memory:
    """A piece of device memory that somebody else owns, for ``torch.as_tensor``."""

    def __init__(self, ptr, count, typestr):
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (ptr, False),
                                         "version": 2, "strides": None}


def _view(owner, ptr: int, count: int, dtype) -> torch.Tensor:
    """A tensor over a stage executor's memory; it keeps the executor, whose end would free it."""
    t = torch.as_tensor(_Memory(ptr, count, "<f4" if dtype is torch.float32 else "<i2"), device="cuda")
    t = t if dtype is torch.float32 else t.view(dtype)
    t.owner = owner
    return t


class _Row:
    def __init__(self, c, seed):
        self.c, self.spec, self.dtype = c, _spec(c), DTYPES[c["dtype"]]
        self.plan = make_rank_plan(_schedule(c), c["n"], c["rank"])
        self.ex = rt.StageExecutor(self.spec, self.plan.n_chunks, c["layers"], self.plan.max_live,
                                   self.plan.split_backward, True, False, c["group"])
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        self.layers = []
        for chunk in range(self.plan.n_chunks):
            for layer in range(c["layers"]):
                self.layers.append((chunk, layer))
                for name, rows, cols in self.ex.params:
                    p = self._of(rt.load().jpp_stage_param_ptr, chunk, layer, name, rows * cols, self.dtype)
                    # weights as an initialised model has them, the router's wide enough to
                    # choose, gains near one and small offsets as after some training
                    std = 0.1 if name.endswith("_g") else self.spec.hidden ** -0.5 if name == "Wr" else 0.02
                    for i in range(0, p.numel(), 1 << 27):
                        q = p[i:i + (1 << 27)]
                        v = torch.randn(q.numel(), generator=gen, device="cuda") * std
                        q.copy_(v + 1 if name.endswith("_g") else v)
        shape = (self.plan.n_chunks, c["n"], self.spec.tokens, self.spec.hidden)
        self.x, self.dy = (torch.empty(shape, dtype=self.dtype, device="cuda") for _ in range(2))
        for t in (self.x, self.dy):
            for i in range(shape[0]):
                for j in range(shape[1]):
                    t[i, j] = torch.randn(shape[2:], generator=gen, device="cuda")
        self.y, self.dx = torch.zeros_like(self.x), torch.zeros_like(self.dy)
        self.addr = {(fwd, i, j): (a[i, j].data_ptr(), b[i, j].data_ptr())
                     for fwd, a, b in ((True, self.x, self.y), (False, self.dy, self.dx))
                     for i in range(shape[0]) for j in range(shape[1])}
        self.loop = RankLoop(self.ex, self.plan, overlap_fused=False)
        self.step = 0
        if c["adam"]:
            self.ex.optimizer_init()
        self.result = {"y": self.y, "dx": self.dx, **self._state()}
        self.graph = None
        if c["graph"]:
            torch.cuda.synchronize()
            stream = rt.Stream()
            self.enqueue(stream.ptr)          # first launches configure their kernels
            stream.sync()
            self.ex.quiesce()
            self.graph = rt.Graph(stream)
            with self.graph:
                self.enqueue(stream.ptr)

    def _of(self, fn, chunk, layer, name, count, dtype):
        import ctypes
        p = ctypes.c_void_p()
        rt.check(fn(self.ex.handle, chunk, layer, self.ex.index[name], ctypes.byref(p)))
        return _view(self.ex, p.value, count, dtype)

    def _state(self):
        """The layers' gradients, or with an update behind the loop their parameters and
        moments; a layer's tensors lie one behind the other."""
        lib = rt.load()
        count = sum(r * k for _, r, k in self.ex.params)
        first = self.ex.params[0][0]
        out = {}
        for chunk, layer in self.layers:
            key = f"{chunk}/{layer}"
            if not self.c["adam"]:
                out["grad " + key] = self._of(lib.jpp_stage_grad_ptr, chunk, layer, first, count,
                                              torch.float32)
                continue
            out["param " + key] = self._of(lib.jpp_stage_param_ptr, chunk, layer, first, count, self.dtype)
            for which, what in enumerate(("weight ", "m ", "v ")):
                if which == 0 and self.c["dtype"] == "f32":
                    continue
                out[what + key] = self._of(lambda h, c, li, i, p: lib.jpp_stage_opt_ptr(h, which, c, li, i, p),
                                           chunk, layer, first, count, torch.float32)
        return out

    def io(self, pt, lane):
        return self.addr[pt.exec_kind is TaskType.FWD, pt.chunk, pt.task.mubatch_idx]

    def enqueue(self, stream=None):
        self.ex.zero_grads(stream)
        self.loop.run(self.io, stream=stream)
        self.ex.join(stream)

    def run(self):
        if self.graph is not None:
            self.graph.launch(0)
        else:
            self.enqueue()
        if self.c["adam"]:
            self.step += 1
            self.ex.adam_step(self.step, lr=1e-5, grad_scale=1.0 / self.c["n"])
        return self.result


class _Step:
    def __init__(self, c, seed):
        spec = _spec(c)
        n = c["n"]
        model = jaxpp.nn.TransformerStack(spec, n_layers=c["layers"] * c["stages"],
                                          layers_per_stage=c["layers"])
        ranks = c["mpmd"] or c["stages"]
        mesh = jaxpp.MpmdMesh(jaxpp.DeviceMesh(np.arange(ranks).reshape(ranks, 1), ("stages", "data")),
                              "stages")
        optimizer = jaxpp.optim.adam(1e-3)
        schedule = _schedule(c)

        def loss_fn(params, ubatch):
            out = model.apply(params, ubatch)
            return jaxpp.nn.mse_loss(out, ubatch) / n, out

        @partial(jaxpp.mpmd_jit_with_loop, mpmd_mesh=mesh)
        def train_step(opt_state, params, batch):
            ubatch_grad = partial(jaxpp.value_and_grad(loss_fn, has_aux=True), params)
            (losses, preds), grad = jaxpp.treduce(ubatch_grad, batch, schedule=schedule)
            updates, opt_state = optimizer.update(grad, opt_state, params)
            return opt_state, jaxpp.optim.apply_updates(params, updates), losses, preds

        self.params = model.init(seed=seed, perturb=True)
        rng = np.random.default_rng(seed)
        shape = (n, spec.tokens, spec.hidden)
        # a step in the course of training: the moments hold two earlier batches' gradients (with
        # none the first update is the sign of the gradient)
        opt_state = optimizer.init(self.params)
        for _ in range(2):
            opt_state, *_ = train_step(opt_state, self.params, rng.standard_normal(shape, dtype=np.float32))
        self.train_step, self.opt_state = train_step, opt_state
        self.batch = rng.standard_normal(shape, dtype=np.float32)

    def run(self):
        _, params, losses, preds = self.train_step(self.opt_state, self.params, self.batch)
        return {"params": params, "losses": losses, "preds": preds}


def prepare(case, seed):
    return (_Step if case["kind"] == "step" else _Row)(case, seed)


def run(state):
    return state.run()
