"""GPU: radix selects with refined digits (the default) against the same call
with plain ones (level2 = -1) and the oracle: digit windows as wide as the key
and narrower, keys outside the sampled window on both sides, crowded digits,
one value in much of the vector (second level), the default budget and the
narrowest and widest digits, at the shortest engine length and past it, alone
and as segments of a batch."""
import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu


def _x(W, dt, fam, n):
    f = np.dtype(dt).kind == "f"
    if fam == "wide":
        return W.normal_f64(11, n).astype(dt) if f else W.uint_range(11, n, 0, 2**32 - 1).view(dt)
    base = W.uint_range(11, n, 1 << 20, (1 << 20) + (1 << 14)).astype(np.int64)
    if fam == "narrow":  # a few keys far below and far above a narrow window
        base[[3, n // 2, n - 1]] = [1, 2, (1 << 31) - 1]
    elif fam == "spike":  # a tenth of the vector is one value, the rest in two lumps
        base[W.uint_range(12, n, 0, 9) == 0] = (1 << 20) + 77
        base[W.uint_range(13, n, 0, 2) == 0] += 1 << 29
    return base.astype(dt)


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.uint32, np.int32])
@pytest.mark.parametrize("fam", ["wide", "narrow", "spike"])
def test_refined_digits(pkg, O, dtype, fam):
    W = pkg.workloads
    ctx = pkg.Context(0)
    for n in (65536 // np.dtype(dtype).itemsize + 1, 300_003, 1_500_000):
        x = _x(W, dtype, fam, n)
        d = pkg.DeviceArray.from_host(x)
        k = np.concatenate([W.k_uniform(14, n, 200, dedup=False), [1, 2, 3, n // 2, n - 1, n]]).astype(np.uint32)
        want = bits(O.sort_choose(x, k))
        for rb in (0, 4, 14):
            for l2 in (0, 1, -1):
                print(f"refine {np.dtype(dtype).name} {fam} n={n} radix_bits={rb} level2={l2}", flush=True)
                got = pkg.multiselect(d, k, ctx, kind="radix", radix_bits=rb, level2=l2)
                assert np.array_equal(bits(got), want), (n, rb, l2)
        table = pkg.segment_table([n // 2, n - n // 2, n // 3], ["radix", "bucket", "radix"], [50, 3, 50],
                                  offsets=[0, n // 2, 5])
        m = [n // 2, n - n // 2, n // 3]
        ks = [W.k_uniform(15 + i, v, q, dedup=False).astype(np.uint32) for i, (v, q) in enumerate(zip(m, (50, 3, 50)))]
        b = pkg.Batch(dtype, table, np.concatenate(ks))
        parts = [x[:m[0]], x[m[0]:], x[5:5 + m[2]]]
        assert np.array_equal(bits(b(d)), bits(np.concatenate([O.sort_choose(v, kk) for v, kk in zip(parts, ks)])))
        b.close()
        d.free()
    ctx.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.uint32, np.int32])
def test_short_radix_and_single_key_digits(pkg, O, dtype):
    """Radix selects of short vectors (cut by their sample) and of long ones
    whose sampled window has a digit per key, with a few keys outside it."""
    W = pkg.workloads
    ctx = pkg.Context(0)
    eb = np.dtype(dtype).itemsize
    for n in (16385, 100003, (1 << 24) // eb - 1, (1 << 24) // eb, (1 << 24) // eb + 9):
        for narrow in (False, True):
            x = W.uint_range(n % 89, n, 0, 1023 if narrow else 2**32 - 1)
            x = x.view(dtype) if np.dtype(dtype).kind != "f" and not narrow else x.astype(dtype)
            if narrow:  # keys that no sample is likely to hold
                x[[5, n // 2, n - 3]] = np.array([1 << 20, 1500, 2000]).astype(dtype)
                if dtype != np.uint32:
                    x[7] = -9
            d = pkg.DeviceArray.from_host(x)
            for k in (np.array([1, 2, 3, 4, n // 2, n - 1, n]), np.arange(n // 3, n // 3 + 400)):
                for opts in ({}, {"seed": 5}, {"level2": -1}, {"level2": 1}, {"radix_bits": 11}):
                    print(f"radix {np.dtype(dtype).name} n={n} narrow={narrow} nk={k.size} {opts}", flush=True)
                    kk = k.astype(np.uint32)
                    got = pkg.multiselect(d, kk, ctx, kind="radix", **opts)
                    assert np.array_equal(bits(got), bits(O.sort_choose(x, kk)))
            d.free()
    ctx.close()
