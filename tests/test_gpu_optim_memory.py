"""Host memory of the optimizer step over host arrays: what it takes besides its results and what
its results keep alive, and that leaves update alike however they travel."""
import tracemalloc

import numpy as np
import pytest

from jaxpp_amd import optim
from jaxpp_amd import runtime as rt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    rt.require_gpu()


def tree(rng, shapes):
    return {f"p{i}": rng.standard_normal(s, dtype=np.float32) for i, s in enumerate(shapes)}


def test_a_large_leaf_is_not_packed_on_the_host():
    """A leaf beyond a run's size is uploaded from its own memory: the step's host arrays are its
    results (update and moments; the sum) and nothing as large beside them."""
    rng = np.random.default_rng(0)
    shape = (1 + rt.COPY_RUN // 1024, 1024)
    nbytes = 4 * shape[0] * shape[1]
    grads, params, opt = tree(rng, [shape]), tree(rng, [shape]), optim.adam(1e-3)
    state = opt.init(params)
    print(f"leaf of {shape}", flush=True)
    tracemalloc.start()
    updates, state = opt.update(grads, state, params)
    peak = tracemalloc.get_traced_memory()[1]
    tracemalloc.reset_peak()
    before = tracemalloc.get_traced_memory()[0]
    new = optim.apply_updates(params, updates)
    peak_sum = tracemalloc.get_traced_memory()[1] - before
    tracemalloc.stop()
    assert peak <= 3.1 * nbytes and peak_sum <= 1.1 * nbytes, (peak / nbytes, peak_sum / nbytes)
    np.testing.assert_array_equal(new["p0"], params["p0"] + updates["p0"])


@pytest.mark.parametrize("shapes", [[(1 + rt.COPY_RUN // 64, 64)], [(1000, 7)] * 40 + [(3,), ()]], ids=["large", "run"])
def test_the_state_does_not_keep_the_updates(shapes):
    rng = np.random.default_rng(1)
    grads, opt = tree(rng, shapes), optim.adam(1e-3)
    state = opt.init(grads)
    nbytes = sum(4 * (a.size + 16) for a in grads.values())
    tracemalloc.start()
    updates, state = opt.update(grads, state)
    del updates
    kept = tracemalloc.get_traced_memory()[0]
    tracemalloc.stop()
    assert set(state) == {"count", "mu", "nu"}
    assert kept <= 2.1 * nbytes + 65536, kept / nbytes


def test_leaves_update_alike_in_runs_and_alone():
    """A leaf by itself (beyond a run's size) and the same values in rows of small leaves: the same
    bits; moments of another type and order of axes than float32 rows among them."""
    rng = np.random.default_rng(2)
    rows, cols = 1 + rt.COPY_RUN // 512, 512
    g, m, v = (rng.standard_normal((rows, cols), dtype=np.float32) for _ in range(3))
    v = np.abs(v)
    opt = optim.adam(1e-3)
    one = opt.update({"a": g}, {"count": 3, "mu": {"a": np.asfortranarray(m)}, "nu": {"a": v.astype(np.float64)}})
    cut = lambda a: [np.array(r) for r in np.array_split(a, 100)]
    many = opt.update(cut(g), {"count": 3, "mu": cut(m), "nu": cut(v)})
    join = lambda t: np.concatenate(t)
    np.testing.assert_array_equal(one[0]["a"], join(many[0]))
    np.testing.assert_array_equal(one[1]["mu"]["a"], join(many[1]["mu"]))
    np.testing.assert_array_equal(one[1]["nu"]["a"], join(many[1]["nu"]))
