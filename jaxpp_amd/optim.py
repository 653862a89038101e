"""The step behind the loop: the optimizer applied to what ``treduce`` returns.

The reference's train step ends with

    updates, opt_state = optimizer.update(grad, opt_state, pars)
    new_pars = optax.apply_updates(pars, updates)

(README.md:90-93; examples/basic.py:234 builds ``optimizer`` with ``optax.adam``).  ``adam``
here has optax's interface - ``init``, ``update`` - and ``apply_updates`` adds the updates;
both run on the GPU (``jpp_adam_step``, ``jpp_grad_accum_f32``), leaf by leaf over pytrees of
float32 host arrays, in the arithmetic ``optax.adam`` uses: f32 tensors, every scalar formed in
double and rounded once.
"""
from __future__ import annotations

from dataclasses import dataclass

import numpy as np

from jaxpp_amd import tracing


def _zip_map(f, *trees):
    a = trees[0]
    if isinstance(a, (tuple, list)):
        return type(a)(_zip_map(f, *ts) for ts in zip(*trees))
    if isinstance(a, dict):
        return {k: _zip_map(f, *(t[k] for t in trees)) for k in a}
    return f(*trees)


def _offsets(leaves):
    """Places of a run's leaves in one vector, each on 64 bytes, and the vector's length."""
    at, n = [], 0
    for a in leaves:
        at.append(n)
        n += -(-a.size // 16) * 16
    return at, n


def _map_runs(f, *trees):
    """A tree like the first of what ``f`` returns per leaf.  ``f`` takes the leaves of a run
    (`runtime.copy_runs`), one list per tree, float32 and contiguous: leaf by leaf a step of four
    small layers was 250 uploads and 200 downloads, and those 20 of its 24 ms."""
    from jaxpp_amd import runtime as rt
    leaves = []
    _zip_map(lambda *ls: leaves.append([np.ascontiguousarray(a, dtype=np.float32) for a in ls]), *trees)
    out = []
    for first, last in rt.copy_runs([ls[0].size for ls in leaves]):
        for ls in leaves[first:last]:
            assert all(a.size >= ls[0].size for a in ls), [a.shape for a in ls]
        out += f(*([ls[k] for ls in leaves[first:last]] for k in range(len(trees))))
    results = iter(out)
    return _zip_map(lambda *_: next(results), *trees)


@dataclass(frozen=True)
class adam:
    """``optax.adam(learning_rate, b1, b2, eps)``: no weight decay, bias-corrected moments."""

    learning_rate: float
    b1: float = 0.9
    b2: float = 0.999
    eps: float = 1e-8

    def init(self, params) -> dict:
        zeros = lambda a: np.zeros(np.shape(a), np.float32)
        return {"count": 0, "mu": tracing.tree_map(zeros, params),
                "nu": tracing.tree_map(zeros, params)}

    def update(self, grads, state: dict, params=None):
        """-> (updates, new state); ``updates = -lr * m_hat / (sqrt(v_hat) + eps)``."""
        from jaxpp_amd import runtime as rt
        rt.require_gpu()
        step = int(state["count"]) + 1

        def run(gs, ms, vs):
            """The leaves of a run as one vector: gradients, moments and updates of `n` elements
            each behind one another on the device, one copy each way."""
            at, n = _offsets(gs)
            host = np.empty(3 * n, np.float32)
            for k, leaves in enumerate((gs, ms, vs)):
                for i, a in enumerate(leaves):
                    host[k * n + at[i]:k * n + at[i] + gs[i].size] = a.reshape(-1)[:gs[i].size]
            buf = rt.DeviceBuffer(16 * n)
            buf.upload(host)
            # weights that start at zero end as the update itself
            rt.check(rt.load().jpp_fill_u32(buf.ptr + 12 * n, 0, n, None))
            rt.adam_step(n, buf.ptr, buf.ptr + 4 * n, buf.ptr + 8 * n, step, master=buf.ptr + 12 * n,
                         lr=self.learning_rate, b1=self.b1, b2=self.b2, eps=self.eps)
            rt.sync()
            out = buf.download(np.float32, (3 * n,), 4 * n)
            part = lambda k, i: out[k * n + at[i]:k * n + at[i] + gs[i].size].reshape(gs[i].shape)
            return [(part(2, i), part(0, i), part(1, i)) for i in range(len(gs))]

        trio = _map_runs(run, grads, state["mu"], state["nu"])
        pick = lambda k: _zip_map(lambda g, t: t[k], grads, trio)
        return pick(0), {"count": step, "mu": pick(1), "nu": pick(2)}


def apply_updates(params, updates):
    """``optax.apply_updates``: ``params + updates``, leaf by leaf, in f32 on the GPU."""
    from jaxpp_amd import runtime as rt
    rt.require_gpu()

    def run(ps, us):
        at, n = _offsets(ps)
        host = np.empty(2 * n, np.float32)
        for k, leaves in enumerate((ps, us)):
            for i, a in enumerate(leaves):
                host[k * n + at[i]:k * n + at[i] + ps[i].size] = a.reshape(-1)[:ps[i].size]
        buf = rt.DeviceBuffer(8 * n)
        buf.upload(host)
        rt.check(rt.load().jpp_grad_accum_f32(None, buf.ptr, buf.ptr + 4 * n, n, 1))
        rt.sync()
        out = buf.download(np.float32, (n,))
        return [out[at[i]:at[i] + p.size].reshape(p.shape) for i, p in enumerate(ps)]

    return _map_runs(run, params, updates)
