"""Host memory of the parameter and gradient copies of many layers: arrays that are reordered or converted on the way
are there some at a time, not for every layer at once."""
import tracemalloc
from types import SimpleNamespace

import numpy as np
import pytest

from jaxpp_amd import runtime as rt

LAYERS, H, F = 12, 256, 2048
PARAMS = [("rms1_g", 1, H), ("Wqkv", H, 3 * H), ("Wo", H, H), ("rms2_g", 1, H), ("Wgu", H, 2 * F), ("Wd", F, H)]
SIZES = [r * c for _, r, c in PARAMS]
LAYER_BYTES = 4 * sum(SIZES)                  # 9.4 MB, of which 4 MB are reordered


def executor(monkeypatch):
    """A stage of the library's shape without a device: tensors at the places a layer's have."""
    lib = SimpleNamespace(jpp_stage_param_ptr="param", jpp_stage_grad_ptr="grad")
    monkeypatch.setattr(rt, "load", lambda: lib)
    ex = rt.StageExecutor.__new__(rt.StageExecutor)
    ex.spec, ex.dtype, ex.params, ex.handle = SimpleNamespace(family="llama"), "f32", PARAMS, None
    monkeypatch.setattr(rt.StageExecutor, "join", lambda self: None)
    at = np.cumsum([0] + SIZES[:-1])
    monkeypatch.setattr(rt.StageExecutor, "_layer_ptrs",
                        lambda self, fn, chunk, layer: [layer * LAYER_BYTES + 4 * int(a) for a in at])
    return ex


def peak(f):
    tracemalloc.start()
    try:
        out = f()
        size, most = tracemalloc.get_traced_memory()
        return out, size, most
    finally:
        tracemalloc.stop()


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["reordered", "converted"])
def test_set_params_of_many_layers(monkeypatch, dtype):
    ex = executor(monkeypatch)
    rng = np.random.default_rng(0)
    host = {n: rng.standard_normal((r, c)).astype(dtype) for n, r, c in PARAMS}
    want = {n: a.astype(np.float32).reshape(-1) for n, a in host.items()}
    want["Wgu"] = want["Wgu"].reshape(H, 2 * F)[:, ex._device_columns("Wgu", 2 * F)].reshape(-1)
    seen = []

    def copy_in(items, bf16=False):
        for (a, ptr) in items:
            layer, rest = divmod(ptr, LAYER_BYTES)
            name = PARAMS[[4 * sum(SIZES[:i]) for i in range(len(SIZES))].index(rest)][0]
            assert np.array_equal(a.reshape(-1), want[name])
            seen.append((layer, name))

    monkeypatch.setattr(rt, "copy_in", copy_in)
    _, _, most = peak(lambda: rt.set_params([(ex, 0, li, host) for li in range(LAYERS)]))
    assert sorted(seen) == sorted((li, n) for li in range(LAYERS) for n, _, _ in PARAMS)
    # a batch, the tensor that did not fit into it and its copy on the way
    assert most <= 4 * rt.COPY_BATCH + 3 * 4 * max(SIZES), most


def test_get_grads_of_many_layers(monkeypatch):
    ex = executor(monkeypatch)

    def copy_out(items, bf16=False):
        for a, ptr in items:
            a[:] = np.arange(ptr // 4, ptr // 4 + a.size) % 65536

    monkeypatch.setattr(rt, "copy_out", copy_out)
    out, size, most = peak(lambda: rt.get_grads([(ex, 0, li) for li in range(LAYERS)]))
    for li, g in enumerate(out):
        at = li * LAYER_BYTES // 4
        for (name, rows, cols), n in zip(PARAMS, SIZES):
            want = (np.arange(at, at + n) % 65536).astype(np.float32).reshape(rows, cols)
            at += n
            if name == "Wgu":
                back = np.empty_like(want)
                back[:, ex._device_columns(name, cols)] = want
                want = back
            assert np.array_equal(g[name].reshape(rows, cols), want), (li, name)
    # beside the results: of a batch the tensors that leave it reordered, and what makes one of them
    assert most - size <= 4 * rt.COPY_BATCH // 2 + 4 * 4 * max(SIZES), (most, size)
