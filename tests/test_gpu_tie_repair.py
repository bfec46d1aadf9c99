"""Sorts of 8-byte keys that leave low digits to the repair of ties: keys as they
come, for which the sort decides how many digits that is, and, with the number
forced, runs of ties of every length that the repair treats differently."""
import numpy as np
import pytest

from conftest import log
from oracle import oracle as o
from test_gpu_radix_sort import same_bits, sort_keys, sort_pairs
from test_gpu_small_sort import rank_path  # noqa: F401  (both ranking paths)

pytestmark = pytest.mark.gpu


def check(k, vdt, descending=False):
    """Sorts k (with values of vdt, None: alone), compares with the oracle; the digits left out."""
    import ctypes

    import gpu_util as g
    from lc_parallel_primitive_amd import DeviceRadixSort, lib

    n, name = k.size, k.dtype.name
    dk, ko, s = g.to_dev(k), g.empty(k.size, k.dtype), DeviceRadixSort()
    if vdt is None:
        tmp = g.temp(s.GetSortKeysTempStorageBytes(name, n))
        (s.SortKeysDescending if descending else s.SortKeys)(tmp, dk, ko, n)
        assert same_bits(g.to_host(ko), o.radix_sort(k, descending=descending, nthreads=8))
    else:
        v = np.arange(n).astype(vdt)
        tmp = g.temp(s.GetSortPairsTempStorageBytes(name, np.dtype(vdt).name, n))
        vo = g.empty(n, vdt)
        (s.SortPairsDescending if descending else s.SortPairs)(tmp, dk, ko, g.to_dev(v), vo, n)
        rk, rv = o.radix_sort(k, v, descending=descending, nthreads=8)
        assert same_bits(g.to_host(ko), rk) and same_bits(g.to_host(vo), rv)
    digits = ctypes.c_int(-1)
    assert lib().lcpp_test_sort_cut(tmp.data_ptr(), tmp.numel(), ctypes.byref(digits)) == 0
    return digits.value


@pytest.mark.parametrize("n", [8193, 100_003, 2_000_003])
def test_frequent_keys_sort_every_digit(gpu, n):
    """Long runs of ties (one frequent key, few distinct ones, equal keys with
    others of the same upper bits) leave no digit to the repair, where one
    workgroup would have them; keys spread evenly do."""
    rng = np.random.default_rng(n)
    full = rng.integers(0, 1 << 64, n, dtype=np.uint64)
    u = rng.random(n)
    zeros = np.where(u < 0.5, np.uint64(0), full)
    sentinels = np.where(u < 0.3, np.uint64(0), np.where(u > 0.999, np.uint64(1), full))
    few = full[:10][rng.integers(0, 10, n)]
    for name, k in (("zeros", zeros), ("sentinels", sentinels), ("few", few), ("floats", np.where(u < 0.5, 0.0, rng.standard_normal(n)))):
        log(f"tie repair frequent {name} n={n}")
        assert check(k, np.uint32) == 0, name
    assert check(full, np.uint32) >= 4
    assert check(rng.standard_normal(n), None) >= 3


def test_more_keys_than_upper_values_sort_every_digit(gpu):
    """40-bit keys have 2^24 values above 16 bits: two digits are left out of a
    tenth as many keys, none of half as many again, which nearly all tie."""
    rng = np.random.default_rng(4)
    for n, digits in ((1_600_000, 2), (25_000_000, 0)):
        log(f"tie repair 40-bit keys n={n}")
        assert check(rng.integers(0, 1 << 40, n, dtype=np.uint64), None) == digits


@pytest.fixture
def set_cut(gpu):
    import lc_parallel_primitive_amd as lcpp

    yield lcpp.lib().lcpp_test_set_sort_cut
    assert lcpp.lib().lcpp_test_set_sort_cut(-1) == 0


def runs(n, sizes, digits, rng):
    """n uint64 keys in a random order, groups of these sizes equal in the bits above `digits` digits."""
    k = rng.integers(0, 1 << 64, n, dtype=np.uint64)
    low = np.uint64((1 << 8 * digits) - 1)
    at = 0
    while True:
        for size in sizes:
            if at + size > n:
                rng.shuffle(k)
                return k
            k[at:at + size] = (k[at] & ~low) | (k[at:at + size] & low)
            at += size


RUNS = {"pairs": [2, 1, 3], "short": [31, 32, 33, 34, 1], "ranked": [64, 65, 1, 255, 256, 257, 2],
        "digits": [256, 257, 300, 900, 1], "LDS edge": [2111, 2112, 2113], "chunks": [1023, 4096, 1, 4097],
        "long": [20_001, 7]}


@pytest.mark.parametrize("layout", RUNS)
@pytest.mark.parametrize("vdt", [None, np.uint32, np.int64])
def test_runs_of_every_length(set_cut, layout, vdt):
    """Runs of ties at the lengths that the repair treats differently, differing
    in two, three and five digits, whatever the rule would say to them."""
    for digits in (2, 3, 5):
        assert set_cut(digits) == 0
        rng = np.random.default_rng(digits)
        for n in (40_000, 100_003):
            k = runs(n, RUNS[layout], digits, rng)
            for descending in (False, True):
                log(f"tie repair runs {layout} n={n} values={vdt} digits={digits} desc={descending}")
                assert check(k, vdt, descending) == digits
            kk = k.view(np.int64) if digits == 3 else np.where(np.isnan(k.view(np.float64)), 0.5, k.view(np.float64))
            assert check(kk, vdt, digits == 5) == digits
    # equal keys: runs in order already, and one key out of order in the longest
    k = np.repeat(rng.integers(0, 1 << 64, 1 + 40_000 // 500, dtype=np.uint64), 500)[:40_000]
    k[:20_000] = k[0] | np.uint64(1)
    k[19_000] ^= np.uint64(1)
    assert check(k, vdt) == 5


def layouts(n, rng):
    """name -> n uint64 sort keys"""
    full = rng.integers(0, 1 << 64, n, dtype=np.uint64)
    out = {"uniform": full}
    # groups of equal upper 40 bits, of every length: too many for a digit to be left out
    k = full.copy()
    at = 0
    for size in (2, 2, 3, 31, 32, 33, 34, 64, 65, 100, 257, 900, 2111, 2112, 2113, 4097, 6000):
        if at + size > n // 4:
            break
        low = rng.integers(0, 1 << 24, size, dtype=np.uint64)
        k[at:at + size] = (full[at] & ~np.uint64(0xFFFFFF)) | low
        at += size
    rng.shuffle(k)
    out["clusters"] = k
    dup = full.copy()
    dup[rng.random(n) < 0.3] = dup[7]  # one frequent key: its run is in order already
    out["duplicates"] = dup
    # few values per byte, no run short: every digit needs its pass
    bits = rng.integers(0, 2, (n, 8), dtype=np.uint8)
    out["few"] = bits.view(np.uint64).reshape(n).copy()
    out["dense"] = np.arange(n, dtype=np.uint64)[::-1].copy() * np.uint64(0x10001)
    out["sorted"] = np.sort(full)
    return out


@pytest.mark.parametrize("n", [8193, 40_000, (1 << 19) + 1, 1_500_000])
@pytest.mark.parametrize("vdt", [None, np.uint32, np.int64])
def test_uint64_layouts(rank_path, n, vdt):  # noqa: F811
    import gpu_util as g

    for name, k in layouts(n, np.random.default_rng(n)).items():
        for descending in (False, True):
            log(f"tie repair {name} n={n} values={vdt} desc={descending}")
            if vdt is None:
                got = g.to_host(sort_keys(g.to_dev(k), n, np.uint64, descending=descending))
                assert same_bits(got, o.radix_sort(k, descending=descending, nthreads=8)), name
            else:
                v = np.arange(n).astype(vdt)
                rk, rv = o.radix_sort(k, v, descending=descending, nthreads=8)
                ko, vo = sort_pairs(g.to_dev(k), g.to_dev(v), n, np.uint64, vdt, descending)
                assert same_bits(g.to_host(ko), rk) and same_bits(g.to_host(vo), rv), name


@pytest.mark.parametrize("kdt", [np.int64, np.float64])
@pytest.mark.parametrize("n", [8193, 300_001, 1_200_000])
def test_signed_and_floating(gpu, kdt, n):
    import gpu_util as g

    rng = np.random.default_rng(n)
    if kdt == np.int64:
        k = rng.integers(-(1 << 63), 1 << 63, n, dtype=np.int64)
    else:
        k = rng.standard_normal(n)
        k[::97], k[1::101] = 0.0, -0.0
        k[2::103] = rng.standard_normal(k[2::103].size) * 1e-310  # around zero, equal upper bits
        k[3:7] = [np.inf, -np.inf, 5e-324, -5e-324]
    v = np.arange(n, dtype=np.uint32)
    for descending in (False, True):
        rk, rv = o.radix_sort(k, v, descending=descending, nthreads=8)
        ko, vo = sort_pairs(g.to_dev(k), g.to_dev(v), n, kdt, np.uint32, descending)
        assert same_bits(g.to_host(ko), rk) and same_bits(g.to_host(vo), rv)


def test_output_over_input(gpu):
    """Sorting in place takes the even number of passes that it always took."""
    import gpu_util as g
    from lc_parallel_primitive_amd import DeviceRadixSort

    n = 100_003
    k = np.random.default_rng(1).integers(0, 1 << 64, n, dtype=np.uint64)
    v = np.arange(n, dtype=np.uint32)
    dk, dv = g.to_dev(k), g.to_dev(v)
    tmp = g.temp(DeviceRadixSort.GetSortPairsTempStorageBytes("uint64", "uint32", n))
    DeviceRadixSort().SortPairs(tmp, dk, dk, dv, dv, n)
    rk, rv = o.radix_sort(k, v)
    assert same_bits(g.to_host(dk), rk) and same_bits(g.to_host(dv), rv)


@pytest.mark.parametrize("keys_over_values", [False, True])
def test_output_over_the_other_input(gpu, keys_over_values):
    """keys_out over vals_in, or vals_out over keys_in: uniform keys of this
    number would take three passes, the first of them from the inputs to the
    outputs."""
    import gpu_util as g
    from lc_parallel_primitive_amd import DeviceRadixSort

    n = 100_003
    k = np.random.default_rng(3).integers(0, 1 << 64, n, dtype=np.uint64)
    v = np.arange(n, dtype=np.uint64) * 3
    dk, dv, other = g.to_dev(k), g.to_dev(v), g.empty(n, np.uint64)
    ko, vo = (dv, other) if keys_over_values else (other, dk)
    tmp = g.temp(DeviceRadixSort.GetSortPairsTempStorageBytes("uint64", "uint64", n))
    DeviceRadixSort().SortPairs(tmp, dk, ko, dv, vo, n)
    rk, rv = o.radix_sort(k, v)
    assert same_bits(g.to_host(ko), rk) and same_bits(g.to_host(vo), rv)


def test_graph_replays(gpu):
    """A captured sort plans again for the keys of each replay."""
    import gpu_util as g
    import torch
    from lc_parallel_primitive_amd import DeviceRadixSort

    n = 100_003
    rng = np.random.default_rng(2)
    dk, ko = g.empty(n, np.uint64), g.empty(n, np.uint64)
    tmp = g.temp(DeviceRadixSort.GetSortKeysTempStorageBytes("uint64", n))
    s = DeviceRadixSort()
    s.SortKeys(tmp, dk, ko, n)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        s.SortKeys(tmp, dk, ko, n)
    for name, k in layouts(n, rng).items():
        dk.copy_(torch.from_numpy(k))
        graph.replay()
        assert same_bits(g.to_host(ko), o.radix_sort(k)), name


def test_several_tiles_per_workgroup(set_cut):
    """More tiles than the repair launches workgroups (64 per CU): each takes
    two, with runs at the tiles' edges."""
    n = 64 * 256 * 2048 + 4097
    rng = np.random.default_rng(5)
    k = rng.integers(0, 1 << 64, n, dtype=np.uint64)
    a, b = k[0:n - 2:3], k[1:n - 1:3]  # pairs
    a[:] = (b & ~np.uint64(0xFFFFFFFF)) | (a & np.uint64(0xFFFFFFFF))
    k[5_000_000:5_003_000] = (k[0] & ~np.uint64(0xFFFFFF)) | (k[5_000_000:5_003_000] & np.uint64(0xFFFFFF))
    assert set_cut(4) == 0
    log(f"tie repair several tiles n={n}")
    assert check(k, np.uint32) == 4
