"""GPU: selects whose second pass reads the candidates that the count pass
kept (SEG_SPEC): top-K, clustered ranks and a few ranks, at the shortest
length that predicts and past it, aligned and not; a chunk with more
candidates than its part holds (a sorted vector has them all in one place); a
share of the keys at the limit and past it; duplicates; several sample seeds
(some predict wrongly); a batch of both kinds of segment, replayed.  Every
result against the oracle; the device's own record says which selects read
their candidates."""
import numpy as np
import pytest

from conftest import bits
from invariants import SEGSTATE, read, regions

pytestmark = pytest.mark.gpu

MIN = 1 << 17  # kSpecMinLen


def _x(W, dt, fam, n):
    if np.dtype(dt).kind != "f":
        x = W.uint_range(9, n, 0, 2**32 - 1 if fam == "spread" else 5000).view(dt)
    else:
        x = (W.normal_f32(9, n) if fam != "copies" else np.rint(W.normal_f32(9, n) * 100) + 0).astype(dt)
    return np.sort(x) if fam == "sorted" else x


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.uint32, np.int32])
@pytest.mark.parametrize("fam", ["spread", "sorted", "copies"])
def test_candidates(pkg, O, dtype, fam):
    W = pkg.workloads
    lib = pkg._lib.lib()
    read_them = 0
    for n in (MIN - 1, MIN, MIN + 1, (1 << 21) + 5, (1 << 22) + 5):
        x = _x(W, dtype, fam, n)
        d = pkg.DeviceArray.from_host(x)
        m = n // 2
        for off in (0, 1):
            v, xv, nv = d.view(off, n - off), x[off:], n - off
            cluster = np.concatenate([np.arange(m - 200, m + 200), [1, nv]]).astype(np.uint32)
            print(f"candidates {np.dtype(dtype).name} {fam} n={nv} off={off}", flush=True)
            for kind, k in (("topk", 1), ("topk", 4096), ("topk", nv // 14), ("topk", nv // 9),
                            ("bucket", [m]), ("bucket", [nv]), ("bucket", cluster), ("bucket", cluster[::-1])):
                for seed in (0, 3, 4):
                    ctx = pkg.Context(0)
                    if kind == "topk":
                        got, want = pkg.topk(v, k, ctx, seed=seed), O.topk(xv, k)
                    else:
                        k = np.asarray(k, np.uint32)
                        got, want = pkg.multiselect(v, k, ctx, seed=seed), O.sort_choose(xv, k)
                    assert np.array_equal(bits(got), bits(want))
                    st = read(lib, regions(pkg, ctx).states, SEGSTATE, 1)[0]
                    read_them += int(st["arrive"])
                    assert nv >= MIN or not int(st["arrive"])
                    ctx.close()
        d.free()
    assert fam != "spread" or read_them > 0


def test_candidates_in_a_batch(pkg, O):
    W = pkg.workloads
    rng = np.random.default_rng(5)
    lens = [int(v) for v in rng.integers(1000, 1 << 20, 40)]
    top = [i % 2 == 0 for i in range(40)]
    nk = [min(n, 4096 >> (i % 8)) if t else 1 + i % 3 for i, (n, t) in enumerate(zip(lens, top))]
    xs = [W.normal_f32(30 + i, n) for i, n in enumerate(lens)]
    ks = [None if t else rng.integers(1, n + 1, q).astype(np.uint32) for n, t, q in zip(lens, top, nk)]
    table = pkg.segment_table(lens, ["topk" if t else "bucket" for t in top], nk)
    b = pkg.Batch(np.float32, table, np.concatenate([k for k in ks if k is not None]))
    want = np.concatenate([O.topk(x, q) if t else O.sort_choose(x, k) for x, t, q, k in zip(xs, top, nk, ks)])
    d = pkg.DeviceArray.from_host(np.concatenate(xs))
    for graph in (False, True, True, True):
        print(f"candidates batch graph={graph}", flush=True)
        assert np.array_equal(bits(b(d, graph=graph)), bits(want))
    b.close()
