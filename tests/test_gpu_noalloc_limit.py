"""GPU: the no-allocation entry point at the largest vectors that its fixed
scratch takes (the planner falls back to smaller histogram rows there), for
both key widths."""
import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,n", [(np.float32, 16_000_000), (np.float64, 8_000_000)])
def test_noalloc_near_its_limit(pkg, O, dtype, n):
    from ggks_multiselect_amd import _lib as L
    lib = L.lib()
    d = pkg.generate(dtype, "normal", 3, n)
    k = pkg.workloads.k_uniform(4, n, 1024, dedup=False)
    dk = pkg.DeviceArray.from_host(k)
    out = pkg.DeviceArray(k.size, dtype)
    print(f"noalloc limit {np.dtype(dtype).name} n={n}", flush=True)
    L.check(lib.ggks_bucket_multiselect_noalloc(pkg.api.dtype_code(dtype), d.ptr, n, dk.ptr, k.size, out.ptr,
                                                None, None))
    L.check(lib.ggks_sync())
    assert np.array_equal(bits(out.to_host()), bits(O.sort_choose(d.to_host(), k)))
