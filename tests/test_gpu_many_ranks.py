"""GPU: selects of vectors past 16 MiB with rank counts at and past a quarter
of the default buckets, where the budget grows by a bit: spread and clustered,
bucket and radix, against the oracle."""
import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.uint32])
def test_many_ranks(pkg, O, dtype):
    W = pkg.workloads
    n = (1 << 24) // np.dtype(dtype).itemsize + 77
    x = W.normal_f32(4, n).astype(dtype) if np.dtype(dtype).kind == "f" else W.uint_range(4, n, 0, 2**32 - 1)
    d = pkg.DeviceArray.from_host(x)
    ctx = pkg.Context(0)
    rng = np.random.default_rng(6)
    for nk in (1024, 1025, 2048, 2049, 6000):
        for k in (rng.integers(1, n + 1, nk), np.arange(n // 2, n // 2 + nk)):
            for kind in ("bucket", "radix"):
                print(f"many ranks {np.dtype(dtype).name} nk={nk} {kind}", flush=True)
                kk = k.astype(np.uint32)
                assert np.array_equal(bits(pkg.multiselect(d, kk, ctx, kind=kind)), bits(O.sort_choose(x, kk)))
    d.free()
    ctx.close()
