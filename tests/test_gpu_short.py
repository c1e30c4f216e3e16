"""GPU: selects and batches of short segments (k_front / k_back): lengths at
the edges of a chunk, of the sample sizes and of the 16 MiB limit, aligned and
not; 1, 1024 and 1025 ranks; one value, a heavy value, sorted keys, the lowest
and highest values of the type; the same context over key types of two widths
in turn (equal plan tables); a batch replayed and run in turn.  Every result
against the oracle."""
import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu

FAMS = ("spread", "copies", "heavy", "one", "sorted", "ends")


def _x(W, dt, fam, n):
    dt = np.dtype(dt)
    x = W.normal_f32(n % 97, n).astype(dt) if dt.kind == "f" else W.uint_range(n % 97, n, 0, 2**32 - 1).view(dt)
    if fam == "copies":
        x = (np.rint(x * 8) + 0).astype(dt) if dt.kind == "f" else (x % 50).astype(dt)
    elif fam == "heavy":
        x[::3] = x[0]
    elif fam == "one":
        x[:] = x[0]
    elif fam == "sorted":
        x = np.sort(x)
    elif fam == "ends":
        lo, hi = (-np.inf, np.inf) if dt.kind == "f" else (np.iinfo(dt).min, np.iinfo(dt).max)
        x[::5], x[1::5] = lo, hi
    return x


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.uint32, np.int32])
@pytest.mark.parametrize("fam", FAMS)
def test_short(pkg, O, dtype, fam):
    W = pkg.workloads
    eb = np.dtype(dtype).itemsize
    limit = (1 << 24) // eb
    ctx = pkg.Context(0)
    lens = [65 * 4096 - 1, 1 << 17, (1 << 17) + 1, (1 << 19) + 1]
    lens += [20000, limit - 1, limit] if fam in ("spread", "heavy") else [64 * 4096 + 1]
    for n in lens:
        x = _x(W, dtype, fam, n)
        d = pkg.DeviceArray.from_host(x)
        for off in (0, 1):
            v, xv, nv = d.view(off, n - off), x[off:], n - off
            print(f"short {np.dtype(dtype).name} {fam} n={n} off={off}", flush=True)
            for nk in (1, 2, 1024, 1025):
                k = np.unique(np.linspace(1, nv, nk).astype(np.uint32))[::-1] if nk > 1 else np.array([nv // 2], np.uint32)
                got = pkg.multiselect(v, k, ctx, seed=nk)
                assert np.array_equal(bits(got), bits(O.sort_choose(xv, k)))
            assert np.array_equal(bits(pkg.topk(v, 1000, ctx)), bits(O.topk(xv, 1000)))
        d.free()
    ctx.close()


def test_short_two_widths_in_turn(pkg, O):
    W = pkg.workloads
    n = 64 * 4096
    x = W.normal_f32(3, n)
    k = np.linspace(1, n, 200).astype(np.uint32)
    ctx = pkg.Context(0)
    a, b = pkg.DeviceArray.from_host(x), pkg.DeviceArray.from_host(x.astype(np.float64))
    for _ in range(3):
        for d, h in ((a, x), (b, x.astype(np.float64)), (a, x)):
            assert np.array_equal(bits(pkg.multiselect(d, k, ctx)), bits(O.sort_choose(h, k)))
    ctx.close()


def test_short_batch(pkg, O):
    W = pkg.workloads
    rng = np.random.default_rng(11)
    lens = [40, 3000, 9000, 16385, 20001, 65537, 131073, 600001, 4096 * 9]
    top = [i % 3 == 1 for i in range(len(lens))]
    nk = [min(n, 700) if t else 1 + 13 * i for i, (n, t) in enumerate(zip(lens, top))]
    xs = [_x(W, np.float32, FAMS[i % 6], n) for i, n in enumerate(lens)]
    ks = [None if t else rng.integers(1, n + 1, q).astype(np.uint32) for n, t, q in zip(lens, top, nk)]
    table = pkg.segment_table(lens, ["topk" if t else "bucket" for t in top], nk)
    b = pkg.Batch(np.float32, table, np.concatenate([k for k in ks if k is not None]))
    want = np.concatenate([O.topk(x, q) if t else O.sort_choose(x, k) for x, t, q, k in zip(xs, top, nk, ks)])
    d = pkg.DeviceArray.from_host(np.concatenate(xs))
    for graph in (False, True, False, True, True):
        print(f"short batch graph={graph}", flush=True)
        assert np.array_equal(bits(b(d, graph=graph)), bits(want))
    b.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32])
@pytest.mark.parametrize("fam", ["spread", "copies", "heavy"])
def test_short_many_ranks(pkg, O, dtype, fam):
    """More ranks than a work-group has threads, up to the limit and past it,
    repeated and out of order."""
    W = pkg.workloads
    ctx = pkg.Context(0)
    rng = np.random.default_rng(8)
    for n in (17001, 130001, (1 << 24) // np.dtype(dtype).itemsize - 5):
        x = _x(W, dtype, fam, n)
        d = pkg.DeviceArray.from_host(x)
        for nk in (2047, 4096, 8191, 8192, 8193):
            print(f"short {np.dtype(dtype).name} {fam} n={n} nk={nk}", flush=True)
            k = rng.integers(1, n + 1, nk).astype(np.uint32)
            assert np.array_equal(bits(pkg.multiselect(d, k, ctx)), bits(O.sort_choose(x, k)))
            assert np.array_equal(bits(pkg.topk(d, nk, ctx)), bits(O.topk(x, nk)))
        d.free()
    ctx.close()
