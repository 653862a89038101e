"""Products whose waves stage their own share of the contraction in tiles of 64 rows: too many tiles of
32 rows for the device, at most one of 64 per CU.  Fewer K-steps than waves and than stages,
remainders of both, numbers of tiles that are not a multiple of the 8 XCDs, the last of the range.  The
bounds are those of the 32-row tiles' test."""
import pytest

import test_gpu_gemm_wave as wave
from jaxpp_amd import runtime as rt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(640, 1280, 64), (1152, 896, 192), (128, 8192, 320), (2176, 256, 576), (1152, 768, 1088),
                                   (384, 2688, 832), (4096, 256, 640)], ids=lambda v: str(v))
@pytest.mark.parametrize("kind", ["nn", "nt", "gelu", "dgelu"])
@pytest.mark.parametrize("pad,tanh", [(0, 0), (8, 1)])
def test_wave_products_of_64_rows(kind, m, n, k, pad, tanh):
    with rt.probe("*") as p:
        wave.test_wave_products(kind, m, n, k, pad, tanh)
    own = f"gemm_{'nn' if kind in ('nn', 'gelu') else 'nt'}_wave"
    assert (own in p.classes) == (kind in ("nn", "nt") or k > 512), p.classes
