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

import math
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


def _upload_run(buf, n, at, *kinds):
    """The kinds of leaves of a run (gradients, moments, ...; one list each) behind one another
    into `buf`, a vector of `n` elements per kind: one packed copy, or of a run of one leaf straight
    from the leaves' own memory.  A leaf's kinds are read as far as the first one reaches."""
    if len(at) == 1:
        for k, (a,) in enumerate(kinds):
            buf.upload(a.reshape(-1)[:kinds[0][0].size], 4 * n * k)
        return
    host = np.empty(n * len(kinds), np.float32)
    for k, leaves in enumerate(kinds):
        for i, a in enumerate(leaves):
            size = kinds[0][i].size
            host[k * n + at[i]:k * n + at[i] + size] = a.reshape(-1)[:size]
    buf.upload(host)


def _download_run(buf, n, at, leaves, *kinds):
    """The kinds `kinds` (adjacent ones) of `buf`'s vectors as arrays of the leaves' shapes, one
    list per kind: views of one array, or of a run of one leaf arrays of their own."""
    if len(at) == 1:
        return [[buf.download(np.float32, leaves[0].shape, 4 * n * k)] for k in kinds]
    out = buf.download(np.float32, (n * len(kinds),), 4 * n * kinds[0])
    return [[out[n * k + i:n * k + i + a.size].reshape(a.shape) for i, a in zip(at, leaves)]
            for k in range(len(kinds))]


def _map_runs(f, *trees):
    """A tree like the first of what ``f`` returns per leaf.  ``f`` takes the leaves of a run
    (`runtime.copy_runs`), one list per tree, float32 and contiguous: leaf by leaf a step of four
    small layers was 250 uploads and 200 downloads, and those 20 of its 24 ms."""
    from jaxpp_amd import runtime as rt
    leaves = []
    _zip_map(lambda *ls: leaves.append(ls), *trees)
    out = []
    for first, last in rt.copy_runs([math.prod(np.shape(ls[0])) for ls in leaves]):
        run = [[np.ascontiguousarray(a, dtype=np.float32) for a in ls] for ls in leaves[first:last]]
        for ls in run:
            assert all(a.size >= ls[0].size for a in ls), [a.shape for a in ls]
        out += f(*([ls[k] for ls in run] for k in range(len(trees))))
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
            each behind one another on the device.  The updates come back as memory of their own:
            the moments outlive the step, they do not."""
            at, n = _offsets(gs)
            buf = rt.DeviceBuffer(16 * n)
            _upload_run(buf, n, at, gs, ms, vs)
            # weights that start at zero end as the update itself
            rt.check(rt.load().jpp_fill_u32(buf.ptr + 12 * n, 0, n, None))
            rt.adam_step(n, buf.ptr, buf.ptr + 4 * n, buf.ptr + 8 * n, step, master=buf.ptr + 12 * n,
                         lr=self.learning_rate, b1=self.b1, b2=self.b2, eps=self.eps)
            rt.sync()
            return list(zip(*_download_run(buf, n, at, gs, 3), *_download_run(buf, n, at, gs, 1, 2)))

        trio = _map_runs(run, grads, state["mu"], state["nu"])
        pick = lambda k: _zip_map(lambda g, t: t[k], grads, trio)
        return pick(0), {"count": step, "mu": pick(1), "nu": pick(2)}


def apply_updates(params, updates):
    """``optax.apply_updates``: ``params + updates``, leaf by leaf, in f32 on the GPU."""
    from jaxpp_amd import runtime as rt
    rt.require_gpu()

    def run(ps, us):
        at, n = _offsets(ps)
        buf = rt.DeviceBuffer(8 * n)
        _upload_run(buf, n, at, ps, us)
        rt.check(rt.load().jpp_grad_accum_f32(None, buf.ptr, buf.ptr + 4 * n, n, 1))
        rt.sync()
        return _download_run(buf, n, at, ps, 0)[0]

    return _map_runs(run, params, updates)
