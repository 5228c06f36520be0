"""The planner's sketch and candidate counts on samples whose keys repeat in
every way that its selection distinguishes: one key, fewer distinct keys than
candidates, exactly as many, many keys of the count at which the candidates
end, and no repeats at all.  Against numpy, exactly."""
import numpy as np
import pytest

from tests.test_planner import sketch_numpy

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    return t


CASES = ["one key", "two keys", "63 keys", "64 keys", "65 keys", "ties", "heavy and unique", "unique", "extremes"]


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("n", [1, 3, 4095, 4096, 100003])
@pytest.mark.parametrize("case", CASES)
def test_sketch_selection(pj, oracle, torch, dtype, n, case):
    from partitioned_join_amd import planner
    rng = np.random.default_rng(n)
    lo, hi = np.iinfo(dtype).min, np.iinfo(dtype).max
    pool = np.unique(rng.integers(lo, hi, 300000, dtype=dtype))
    rng.shuffle(pool)
    if case.endswith(("key", "keys")):
        probe = pool[rng.integers(0, {"one": 1, "two": 2}.get(case.split()[0]) or int(case.split()[0]), n)]
    elif case == "ties":  # 2048 keys twice each in the sample
        probe = np.repeat(pool[:max(1, n // 2 + 1)], 2)[:n]
    elif case == "heavy and unique":
        probe = pool[:n].copy() if n <= pool.size else pool[rng.integers(0, pool.size, n)]
        probe[rng.random(n) < 0.3] = pool[-1]
        probe[rng.random(n) < 0.1] = pool[-2]
    elif case == "unique":
        probe = pool[:n]
    else:
        probe = np.array([lo, hi, 0, -1, 1], dtype=dtype)[rng.integers(0, 5, n)]
    n = probe.size
    build = np.arange(777, dtype=dtype)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    feat, cand, cnt = planner.sketch(d(build), d(probe))
    ef, ek, ec = sketch_numpy(oracle, probe, build.size)
    f = feat.cpu().numpy()
    assert np.array_equal(f[:1024], ef[:1024])
    assert np.allclose(f[1024:], ef[1024:], rtol=1e-6, atol=1e-7)
    got = cand.cpu().numpy().view(np.uint64)
    assert np.array_equal(cnt.cpu().numpy().astype(np.int64), ec)
    assert np.array_equal(got, ek)
    exact = planner.candidate_counts(d(probe), cand, cnt).cpu().numpy()
    u = probe.astype(np.int64).view(np.uint64) if dtype == np.int64 else (probe.astype(np.int64) & 0xFFFFFFFF).astype(np.uint64)
    keys, counts = np.unique(u, return_counts=True)
    of = dict(zip(keys.tolist(), counts.tolist()))
    assert exact.tolist() == [of[int(k)] if c else 0 for k, c in zip(ek, ec)]
