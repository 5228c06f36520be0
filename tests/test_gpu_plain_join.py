"""The plain join's own pipeline (csrc/pj_wide.h) where its shape changes: the
build sizes at which a table no longer fits one chunk, at which the chunk
configuration and the number of partitions change, probe sizes around a round
and a scatter tile, with unique and repeated keys, heavy keys on both sides,
payload columns, key columns that are not 16-byte aligned and outputs that do
not fit.  Every join against the oracle's (all values are whole numbers: the
sorted pairs are equal)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    return t


def spread(ids, dtype):
    """Distinct keys of distinct ids over the whole key range."""
    if dtype == np.int32:
        return (ids.astype(np.uint64) * np.uint64(0x2545F491)).astype(np.uint32).view(np.int32)
    return (ids.astype(np.uint64) * np.uint64(0x9E3779B97F4A7C15) + np.uint64(12345)).view(np.int64)


def check(pj, oracle, torch, bk, pk, bp=None, pp=None, uniq=True, plan=None, shift=0):
    """shift: the key columns start that many keys into their buffers."""
    def dev(a):
        if a is None:
            return None
        t = torch.from_numpy(np.concatenate([np.zeros(shift, a.dtype), a])).cuda()
        return t[shift:]
    got = pj.partitioned_join(dev(bk), dev(pk), dev(bp), dev(pp), plan=plan)
    exp = oracle.sort_pairs(oracle.inner_join_cpu(bk, pk, bp, pp, uniq_keys=uniq))
    g = oracle.sort_pairs(got.cpu().numpy())
    assert len(g) == len(exp), (len(g), len(exp))
    assert np.array_equal(g, exp)


# chunk capacities 3072, 6144, 12288 (int32) and 2048, 5120, 10240 (int64) without
# partitions; then 64 partitions; 2^19 + 1: more than the least number of them
SIZES32 = [1, 2, 511, 512, 513, 3071, 3072, 3073, 6144, 6145, 12288, 12289, 131073, (1 << 20) + 1]
SIZES64 = [1, 511, 513, 2047, 2048, 2049, 5120, 5121, 10240, 10241, 98305, 786433]


@pytest.mark.parametrize("dtype,n", [(np.int32, n) for n in SIZES32] + [(np.int64, n) for n in SIZES64])
def test_build_sizes_where_the_shape_changes(pj, oracle, torch, dtype, n):
    rng = np.random.default_rng(n)
    bk = spread(rng.permutation(n), dtype)
    for ns in (1, 3071, 4097, 2 * n + 8191):
        pk = spread(rng.integers(0, 2 * n, ns), dtype)
        check(pj, oracle, torch, bk, pk)
    plan = pj.plan_default(n, ns, bk.itemsize)
    plan.unique_build_keys = 1
    check(pj, oracle, torch, bk, pk, plan=plan)


@pytest.mark.parametrize("dtype,n", [(np.int32, 5000), (np.int32, 400000), (np.int64, 9000), (np.int64, 400000)])
def test_repeated_and_heavy_keys(pj, oracle, torch, dtype, n):
    rng = np.random.default_rng(n + 1)
    # each key 0 to 12 times, one key in a hundredth of the rows on either side
    ids = rng.integers(0, n // 3, n)
    ids[rng.random(n) < 0.002] = 7
    pid = rng.integers(0, n // 2, 3 * n)
    pid[rng.random(3 * n) < 0.01] = 7
    bp = rng.integers(-2**31, 2**31 - 1, n).astype(np.int32)
    pp = rng.integers(-2**31, 2**31 - 1, 3 * n).astype(np.int32)
    check(pj, oracle, torch, spread(ids, dtype), spread(pid, dtype), bp, pp, uniq=False)
    check(pj, oracle, torch, spread(ids, dtype), spread(pid, dtype), bp, None, uniq=False, shift=1)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_one_partition_holds_more_than_a_chunk(pj, oracle, torch, dtype):
    # 30000 rows of one key beside 200000 others: chunks of one key alone, met by few and by no probes
    rng = np.random.default_rng(5)
    ids = np.concatenate([np.full(30000, 11), rng.permutation(200000) + 100])
    rng.shuffle(ids)
    for heavy in (0, 3, 40):
        pid = np.concatenate([np.full(heavy, 11), rng.integers(50, 300000, 250000)])
        rng.shuffle(pid)
        check(pj, oracle, torch, spread(ids, dtype), spread(pid, dtype), uniq=False)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
def test_ragged_tiles_and_unaligned_columns(pj, oracle, torch, dtype, shift):
    rng = np.random.default_rng(40 + shift)
    for n, ns in [(70000, 4095), (70000, 4096 * 7), (99999, 4096 * 64 + 1), (20000, 1)]:
        check(pj, oracle, torch, spread(rng.permutation(n), dtype), spread(rng.integers(0, 2 * n, ns), dtype), shift=shift)


def test_strided_keys_fill_partitions_evenly_enough(pj, oracle, torch):
    # keys that share their low (or high) bits, extreme values among them
    for step in (1, 1 << 10, 1 << 12, 65536, 3 << 13):
        bk = (np.arange(60000, dtype=np.int64) * step).astype(np.uint32).view(np.int32)
        bk = np.unique(bk)
        pk = np.concatenate([bk, bk[::3] ^ 1, np.array([-1, 0, 2**31 - 1, -2**31], np.int32)])
        check(pj, oracle, torch, bk, pk)


@pytest.mark.parametrize("n,ns", [(3000, 9000), (300000, 900000)])
def test_output_that_does_not_fit(pj, oracle, torch, n, ns):
    rng = np.random.default_rng(9)
    bk, pk = spread(rng.permutation(n), np.int32), spread(rng.integers(0, n, ns), np.int32)
    d = lambda a: torch.from_numpy(a).cuda()
    for cap in (0, 1, 4095, ns - 1):
        out = torch.full((cap + 64, 2), -7, dtype=torch.int32, device="cuda")
        count = pj.partitioned_join_async(d(bk), d(pk), out[:cap])
        assert int(count.item()) == ns
        assert bool((out[cap:] == -7).all())  # nothing past the capacity
    out = torch.empty((ns, 2), dtype=torch.int32, device="cuda")
    assert int(pj.partitioned_join_async(d(bk), d(pk), out).item()) == ns
    exp = oracle.sort_pairs(oracle.inner_join_cpu(bk, pk, None, None, uniq_keys=True))
    assert np.array_equal(oracle.sort_pairs(out.cpu().numpy()), exp)


@pytest.mark.parametrize("nb,ns", [((1 << 23) - 1, 1 << 22), (1 << 23, 1 << 22), ((1 << 25) + 1, 1 << 24)])
def test_large_builds_where_the_tag_identifies_the_key(pj, torch, nb, ns):
    """2^23: the int32 keys leave the table (digit, bucket and tag are the
    key); 2^25 + 1: chunks of 16384.  Every probe row with a partner appears
    once, with that partner."""
    g = torch.Generator(device="cuda").manual_seed(nb)
    ids = torch.randperm(nb, generator=g, device="cuda")
    pid = torch.randint(0, 2 * nb, (ns,), generator=g, device="cuda")
    for c in (1, 0x2545F491):
        bk, pk = (ids * c).to(torch.int32), (pid * c).to(torch.int32)
        pairs = pj.partitioned_join(bk, pk).to(torch.int64)
        assert pairs.shape[0] == int((pid < nb).sum())
        assert bool((ids[pairs[:, 0]] == pid[pairs[:, 1]]).all())
        assert torch.unique(pairs[:, 1]).numel() == pairs.shape[0]


@pytest.mark.parametrize("dtype,nb", [("int32", 1 << 24), ("int32", (1 << 24) + 1), ("int32", 1 << 25), ("int64", 4608 * 2048),
                                      ("int64", 4608 * 2048 + 1), ("int64", 9728 * 2048), ("int64", 9728 * 2048 + 1)])
def test_large_builds_around_the_last_doublings_of_the_partitions(pj, torch, dtype, nb):
    """2048 and 4096 partitions and their chunk sizes, average and largest."""
    g = torch.Generator(device="cuda").manual_seed(nb)
    ids = torch.randperm(nb, generator=g, device="cuda")
    pid = torch.randint(0, 2 * nb, (1 << 22,), generator=g, device="cuda")
    spread = (lambda x: (x * 0x2545F491).to(torch.int32)) if dtype == "int32" else (lambda x: x * 0x2545F4914F6CDD1D)
    pairs = pj.partitioned_join(spread(ids), spread(pid)).to(torch.int64)
    assert pairs.shape[0] == int((pid < nb).sum())
    assert bool((ids[pairs[:, 0]] == pid[pairs[:, 1]]).all())
    assert torch.unique(pairs[:, 1]).numel() == pairs.shape[0]


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("step", [3, 4, 8, 24, 128])
def test_small_strides_of_both_key_sizes(pj, oracle, torch, dtype, step):
    rng = np.random.default_rng(step)
    bk = (rng.permutation(150001) * step).astype(dtype)
    pk = (rng.integers(0, 300000, 200003) * step + (rng.random(200003) < 0.1)).astype(dtype)
    check(pj, oracle, torch, bk, pk)
