"""A stage's forward reads its input where the caller has it and keeps a copy for the backward: with the output
in another buffer, over the input, and with an input at an address that vector loads do not take, the
results are the same to the last bit, and the caller may overwrite the input once the forward has run."""
import numpy as np
import pytest

from jaxpp_amd import runtime as rt
from jaxpp_amd.model import LayerSpec, boundary_tensor, init_layer_params
from jaxpp_amd.types import TaskType

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    rt.require_gpu()


def spec(family, h, hd, seq, dtype):
    experts = dict(n_experts=8, top_k=2) if family == "mixtral" else {}
    return LayerSpec(family, h, h // hd, 256, seq, 1, n_kv_heads=h // hd, head_dim=hd, causal=family != "bert",
                     eps=1e-5, dtype=dtype, **experts)


# (a row of the norm is 1 to 16 loads of a lane)
@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("family,h,hd,seq,dtype", [
    ("bert", 128, 64, 128, "bf16"), ("bert", 1152, 128, 256, "bf16"), ("bert", 4352, 128, 128, "bf16"),
    ("decoder", 640, 64, 128, "bf16"), ("llama", 2304, 128, 128, "bf16"), ("mixtral", 256, 128, 128, "bf16"),
    ("bert", 384, 64, 128, "f32"), ("decoder", 128, 64, 256, "f32"), ("llama", 256, 128, 128, "f32")])
def test_forward_reads_its_input_in_place(family, h, hd, seq, dtype, layers):
    s = spec(family, h, hd, seq, dtype)
    shape = (s.tokens, s.hidden)
    es = 4 if dtype == "f32" else 2
    params = [init_layer_params(s, 3, li, perturb=True) for li in range(layers)]
    x, dy = (boundary_tensor(k, 0, 0, shape, 0) for k in ("x", "dy"))
    junk = np.full(shape, 7.0, np.float32)
    results = []
    for way in ("apart", "over the input", "odd address"):
        print(f"stage input {family} {h} {dtype} layers={layers} {way}", flush=True)
        ex = rt.StageExecutor(s, 1, layers, 1, False, True, False, 0)
        for li in range(layers):
            ex.set_params(0, li, params[li])
        src = ex.upload_activation(x)
        big = rt.DeviceBuffer(x.size * es + 16)
        out = src if way == "over the input" else ex.new_activation()
        at = src.ptr
        if way == "odd address":
            at = big.ptr + es
            rt.check(rt.load().jpp_memcpy_d2d_async(at, src.ptr, x.size * es, None))
        ex.run_task(TaskType.FWD, 0, 0, at, out.ptr)
        rt.sync()
        y = ex.download_activation(out, shape)
        if out is not src:      # (else the output has taken its place)
            garbage = ex.upload_activation(junk)
            rt.check(rt.load().jpp_memcpy_d2d_async(at, garbage.ptr, x.size * es, None))
        cot, dx = ex.upload_activation(dy), ex.new_activation()
        ex.run_task(TaskType.BWD, 0, 0, cot.ptr, dx.ptr)
        ex.join()
        rt.sync()
        got = [y, ex.download_activation(dx, shape)]
        for li in range(layers):
            g = ex.get_grads(0, li)
            got += [g[k] for k in sorted(g)]
        ex.close()
        results.append(got)
    for other in results[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(results[0], other))
    assert all(np.isfinite(a).all() and np.abs(a).max() > 0 for a in results[0][:2])
