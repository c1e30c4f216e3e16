"""GPU: synchronous host calls whose k list is read from, and whose outputs
are stored to, pinned host memory in place: output sizes at the limit of the
direct stores (128 KiB) and past it, one output and none to spare, ranks in
random order, on plans of each route (one finisher, short, long); calls of
different routes in turn on one context, so that the staging slots are
reused.  Every result against the oracle."""
import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu

LIMIT = 1 << 17  # kDirectOutBytes


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_host_outputs(pkg, O, dtype):
    W = pkg.workloads
    at = LIMIT // np.dtype(dtype).itemsize
    rng = np.random.default_rng(2)
    ctx = pkg.Context(0)
    vs = [W.normal_f32(n % 13, n).astype(dtype) for n in (3000, 100001, (1 << 22) + 3)]
    ds = [pkg.DeviceArray.from_host(x) for x in vs]
    for nk in (1, 1000, 1024, at - 1, at, at + 1):
        for x, d in zip(vs, ds):
            k = rng.integers(1, x.size + 1, nk).astype(np.uint32)
            for kind in ("bucket", "radix"):
                print(f"host io {np.dtype(dtype).name} n={x.size} nk={nk} {kind}", flush=True)
                got = pkg.multiselect(d, k, ctx, kind=kind)
                assert np.array_equal(bits(got), bits(O.sort_choose(x, k)))
            K = min(nk, x.size)
            assert np.array_equal(bits(pkg.topk(d, K, ctx)), bits(O.topk(x, K)))
    ctx.close()
