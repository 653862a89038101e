"""How a layer's weight gradients leave a stage: which of them by themselves, which in one grid, and
over how many microbatches at once - by the launches counted per kernel class - and that the sums
are those of an ungrouped stage.

Two orders of a sum of n = 2 x 1024 products of random sign differ by about sqrt(n) 2^-24 = 2.7e-6 of the
sum's own size: 1e-5 of the tensor's largest element."""
import numpy as np
import pytest

import parity

from jaxpp_amd import runtime as rt
from jaxpp_amd.model import LayerSpec, boundary_tensor, init_layer_params
from jaxpp_amd.types import TaskType

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    rt.require_gpu()


def run(spec, params, group, n=2):
    """Gradients of n microbatches, and the weight-gradient launches per kernel class that follow
    the last one's backward task (a whole group's, or its own)."""
    shape = (spec.tokens, spec.hidden)
    ex = rt.StageExecutor(spec, 1, 1, n, False, True, False, group)
    ex.set_params(0, 0, params)
    out = ex.new_activation()
    for m in range(n):
        x, dy = (ex.upload_activation(boundary_tensor(k, 0, m, shape)) for k in ("x", "dy"))
        ex.run_task(TaskType.FWD, 0, m, x.ptr, out.ptr)
        if m + 1 < n:
            ex.run_task(TaskType.BWD, 0, m, dy.ptr, out.ptr)
            rt.sync()
            continue
        with rt.probe("*") as p:
            ex.run_task(TaskType.BWD, 0, m, dy.ptr, out.ptr)
            ex.join()
            rt.sync()
    grads = ex.get_grads(0, 0)
    ex.close()
    return grads, {k: v[0] for k, v in p.classes.items() if k.startswith("gemm_tn_")}


W256, MULTI256 = "gemm_tn_accf32_256x256w8", "gemm_tn_accf32_256x256w8_multi"
LLAMA = dict(n_kv_heads=4, head_dim=128, causal=True, rope_theta=5e5, eps=1e-5)


@pytest.mark.parametrize("spec,group,check", [
    # a layer that is not all whole 256x256 tiles: the gate/up gradient (344 of them) by itself and
    # over both microbatches of the group
    (LayerSpec("llama", 2048, 16, 5504, 1024, 1, **LLAMA), 2, lambda c: c[W256] == 1 and MULTI256 not in c),
    # one without a matrix that fills a round: everything in one launch per microbatch
    (LayerSpec("bert", 896, 14, 3584, 128, 1, eps=1e-12), 2,
     lambda c: sum(c.values()) == 2 and all(k.endswith("_multi") for k in c)),
    # 160 whole tiles together: one launch over both microbatches; 90: one for each
    (LayerSpec("bert", 1024, 16, 3072, 128, 1, eps=1e-12), 2, lambda c: list(c.values()) == [1]),
    (LayerSpec("bert", 768, 12, 2304, 128, 1, eps=1e-12), 2, lambda c: list(c.values()) == [2]),
], ids=["wide", "narrow", "half-round", "less"])
def test_weight_gradient_launches(spec, group, check):
    print(f"weight gradients of {spec.family} {spec.hidden}/{spec.ffn}, group {group}", flush=True)
    params = init_layer_params(spec, 3, 0, perturb=True)
    plain, _ = run(spec, params, 0)
    grads, classes = run(spec, params, group)
    assert check(classes), classes
    for name, g in plain.items():
        parity.close(grads[name], g, 1e-5, name)
