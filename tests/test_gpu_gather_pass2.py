"""The gather of payload columns around its workgroup and XCD shares, and the
second partition pass over skewed and ragged pass-1 partitions (its items are
ranges of four scatter tiles).  Whole numbers: equal to numpy's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    return t


@pytest.mark.parametrize("n", [1, 255, 256, 257, 2047, 2048, 2049, 131072 + 1, 512 * 256 * 3 + 77])
def test_gather_sizes(pj, torch, n):
    rng = np.random.default_rng(n)
    pairs = np.stack([rng.integers(0, 5000, n), rng.integers(0, 70000, n)], 1).astype(np.int32)
    b8, p4 = rng.integers(-2**62, 2**62, 5000), rng.integers(-2**31, 2**31 - 1, 70000).astype(np.int32)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    for bcol, pcol in [(b8, p4), (b8.astype(np.int32), p4), (b8, p4.astype(np.int64)), (None, p4), (b8, None)]:
        gb, gp = pj.gather(d(pairs), None if bcol is None else d(bcol), None if pcol is None else d(pcol))
        assert (gb is None) == (bcol is None) and (gp is None) == (pcol is None)
        if bcol is not None:
            assert np.array_equal(gb.cpu().numpy(), bcol[pairs[:, 0]])
        if pcol is not None:
            assert np.array_equal(gp.cpu().numpy(), pcol[pairs[:, 1]])
    # pairs that start at an odd row
    gb, _ = pj.gather(d(pairs)[n // 2:], d(b8), None)
    assert np.array_equal(gb.cpu().numpy(), b8[pairs[n // 2:, 0]])


@pytest.mark.parametrize("kb,b1,b2", [(4, 7, 6), (4, 1, 1), (4, 4, 12), (8, 6, 6), (8, 3, 8)])
@pytest.mark.parametrize("n", [1, 65535, 65537, 700001])
def test_second_pass_over_skewed_partitions(pj, oracle, torch, kb, b1, b2, n):
    rng = np.random.default_rng(n + b1)
    dt = np.int32 if kb == 4 else np.int64
    keys = rng.integers(np.iinfo(dt).min, np.iinfo(dt).max, n, dtype=dt)
    keys[rng.random(n) < 0.5] &= ~((1 << (b1 + b2)) - 1)  # half the rows in partition 0
    keys[rng.random(n) < 0.2] = 12345
    t1, off1 = pj.partition_input_tables_pass_one(torch.from_numpy(keys).cuda(), None, bits=b1, shift=b2)
    t2, off2 = pj.partition_input_tables_pass_two(t1, kb, b1, b2, off1)
    k, p = pj.tuple_keys(t2, kb).cpu().numpy(), pj.tuple_payloads(t2, kb).cpu().numpy()
    oracle.check_partitioned(keys, None, k, p, off2.cpu().numpy().astype(np.int64), 0, b1 + b2)
