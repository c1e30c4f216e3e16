"""GPU: children with many ranks, finished from nearly even bins in LDS
(bin_select), at the edges of its two work-group shapes: 1024 keys (256
threads), 64 KB of keys (1024 threads) and one key past each; a few ranks,
one more than a work-group takes at a time, and every rank; keys spread
evenly, crowded at one end of their range, around zero, in copies of few
values (crowded bins: a wavefront each), in copies of one, and a few bins
holding everything (the sort behind it)."""
import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu


def _values(W, dt, fam, n):
    if fam == "crowded":  # nearly all keys in one coarse bin, most of them distinct
        x = 1.0 + W.uniform_f64(5, n) * 2.0 ** -12
        x[0] = 2.0 ** 40
        return x.astype(dt) if np.dtype(dt).kind == "f" else (x * 2.0 ** 20).astype(np.int64).astype(dt)
    if np.dtype(dt).kind != "f":
        return (W.uint_range(5, n, 0, 2**32 - 1).view(dt) if fam == "even"
                else W.uint_range(5, n, 0, 40).astype(dt))
    if fam == "even":
        return W.uniform_f64(5, n).astype(dt)
    if fam == "tail":
        return W.normal_f64(5, n).astype(dt)
    return np.rint(W.normal_f64(5, n) * 4).astype(dt) + 0  # copies of ~30 values, no -0.0


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.uint32, np.int32])
@pytest.mark.parametrize("fam", ["even", "tail", "copies", "crowded"])
def test_many_ranks_of_one_child(pkg, O, dtype, fam):
    W = pkg.workloads
    cap = 65536 // np.dtype(dtype).itemsize
    ctx = pkg.Context(0)
    for n in (5, 64, 1023, 1024, 1025, 4097, cap - 1, cap):
        x = _values(W, dtype, fam, n)
        d = pkg.DeviceArray.from_host(x)
        for nk in sorted({5, min(n, 33), min(n, 1025), n}):
            print(f"bins {np.dtype(dtype).name} {fam} n={n} {nk} k", flush=True)
            k = (W.splitmix64(nk, 0, nk) % np.uint64(n) + np.uint64(1)).astype(np.uint32) if nk < n \
                else np.arange(1, n + 1, dtype=np.uint32)
            got = pkg.multiselect(d, k, ctx)
            assert np.array_equal(bits(got), bits(O.sort_choose(x, k))), (n, nk)
            got = pkg.topk(d, nk, ctx)
            assert np.array_equal(bits(got), bits(O.topk(x, nk))), (n, nk)
        d.free()
    ctx.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.uint32, np.int32])
@pytest.mark.parametrize("fam", ["lump", "copies", "zero"])
def test_ranks_of_a_child_past_lds(pkg, O, dtype, fam):
    """A child longer than 64 KB of keys, finished window by window: most
    keys in one bucket, spread out in it, in copies of a few values (bins
    longer than LDS, bins that are one value), or around zero (floats crowd
    at both ends of the bucket); one rank, a few, and more than one round of
    them, clustered and spread."""
    W = pkg.workloads
    ctx = pkg.Context(0)
    n = 150_001
    if fam == "copies":
        x = (W.uint_range(6, n, 0, 6).astype(np.int64) * 3 + (W.uint_range(7, n, 0, 99) == 0)).astype(dtype)
    elif fam == "lump" or np.dtype(dtype).kind != "f":
        x = (W.uint_range(6, n, 0, 1 << 18).astype(np.int64) + 5000).astype(dtype)
    else:
        x = (W.normal_f64(6, n) * 1e-20).astype(dtype) + 0
    x[:300] = (np.arange(300, dtype=np.int64) * 7_000_000).astype(dtype)  # the range around the lump
    d = pkg.DeviceArray.from_host(x)
    for k in ([n // 2], [1, 2, n // 3, n // 2, n // 2 + 1, n], np.arange(n // 2, n // 2 + 700),
              W.k_uniform(8, n, 2500, dedup=False)):
        k = np.asarray(k, np.uint32)
        print(f"past LDS {np.dtype(dtype).name} {fam} {k.size} k", flush=True)
        got = pkg.multiselect(d, k, ctx, buckets_log2=8, level2=-1)
        assert np.array_equal(bits(got), bits(O.sort_choose(x, k))), k.size
        got = pkg.topk(d, k.size, ctx, buckets_log2=8, level2=-1)
        assert np.array_equal(bits(got), bits(O.topk(x, k.size))), k.size
    d.free()
    ctx.close()
