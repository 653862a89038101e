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


# Elements of the leaves that go through the device in one go.
BATCH = 1 << 23


def _offsets(leaves):
    """Places of leaves in one vector, one behind the other, and the vector's length (whole 64 bytes)."""
    at, n = [], 0
    for a in leaves:
        at.append(n)
        n += a.size
    return at, -(-n // 16) * 16


def _upload(ptr, n, at, *kinds):
    """The kinds of leaves (gradients, moments, ...; one list each) behind one another to `ptr`, a vector
    of `n` elements per kind, from the leaves' own memory.  A leaf's kinds are read as far as the
    first one reaches."""
    from jaxpp_amd import runtime as rt
    rt.copy_in([(a.reshape(-1)[:first.size], ptr + 4 * (n * k + i))
                for k, leaves in enumerate(kinds) for a, first, i in zip(leaves, kinds[0], at)])


def _download(ptr, n, at, leaves, *kinds):
    """The kinds `kinds` of the vectors at `ptr` as arrays of the leaves' shapes, one list per kind:
    views of one array per kind and run of small leaves (`runtime.copy_runs`)."""
    from jaxpp_amd import runtime as rt
    items, out = [], []
    for k in kinds:
        views = []
        for first, last in rt.copy_runs([a.size for a in leaves]):
            flat = np.empty(at[last - 1] + leaves[last - 1].size - at[first], np.float32)
            items.append((flat, ptr + 4 * (n * k + at[first])))
            views += [flat[i - at[first]:i - at[first] + a.size].reshape(a.shape)
                      for i, a in zip(at[first:last], leaves[first:last])]
        out.append(views)
    rt.copy_out(items)
    return out


def _map_batches(f, *trees):
    """A tree like the first of what ``f`` returns per leaf.  ``f`` takes consecutive leaves of at most
    `BATCH` elements together (or one), one list per tree, float32 and contiguous."""
    leaves = []
    _zip_map(lambda *ls: leaves.append(ls), *trees)
    sizes = [math.prod(np.shape(ls[0])) for ls in leaves]
    out, first = [], 0
    while first < len(leaves):
        last, total = first + 1, sizes[first]
        while last < len(leaves) and total + sizes[last] <= BATCH:
            total += sizes[last]
            last += 1
        batch = [[np.ascontiguousarray(a, dtype=np.float32) for a in ls] for ls in leaves[first:last]]
        for ls in batch:
            assert all(a.size >= ls[0].size for a in ls), [a.shape for a in ls]
        out += f(*([ls[k] for ls in batch] for k in range(len(trees))))
        first = last
    results = iter(out)
    return _zip_map(lambda *_: next(results), *trees)


class _Scratch:
    """Device memory that the batches of one call take in turn."""

    def __init__(self):
        self.buf = None

    def take(self, nbytes: int) -> int:
        from jaxpp_amd import runtime as rt
        if self.buf is None or self.buf.nbytes < nbytes:
            self.buf = None          # (freed before the larger one is taken)
            self.buf = rt.DeviceBuffer(nbytes)
        return self.buf.ptr


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
        scratch = _Scratch()

        def run(gs, ms, vs):
            """The leaves of a batch as one vector: gradients, moments and updates of `n` elements
            each behind one another on the device.  The updates come back as memory of their own:
            the moments outlive the step, they do not."""
            at, n = _offsets(gs)
            ptr = scratch.take(16 * n)
            # weights that start at zero end as the update itself
            rt.check(rt.load().jpp_fill_u32(ptr + 12 * n, 0, n, None))
            _upload(ptr, n, at, gs, ms, vs)
            rt.adam_step(n, ptr, ptr + 4 * n, ptr + 8 * n, step, master=ptr + 12 * n,
                         lr=self.learning_rate, b1=self.b1, b2=self.b2, eps=self.eps)
            return list(zip(*_download(ptr, n, at, gs, 3, 1, 2)))

        trio = _map_batches(run, grads, state["mu"], state["nu"])
        pick = lambda k: _zip_map(lambda g, t: t[k], grads, trio)
        return pick(0), {"count": step, "mu": pick(1), "nu": pick(2)}


def apply_updates(params, updates):
    """``optax.apply_updates``: ``params + updates``, leaf by leaf, in f32 on the GPU."""
    from jaxpp_amd import runtime as rt
    rt.require_gpu()
    scratch = _Scratch()

    def run(ps, us):
        at, n = _offsets(ps)
        ptr = scratch.take(8 * n)
        _upload(ptr, n, at, ps, us)
        rt.check(rt.load().jpp_grad_accum_f32(None, ptr, ptr + 4 * n, n, 1))
        return _download(ptr, n, at, ps, 0)[0]

    return _map_batches(run, params, updates)
