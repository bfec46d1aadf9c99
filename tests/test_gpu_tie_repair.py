"""Sorts of 8-byte keys that leave low digits to the repair of ties: keys whose
upper bits tie in runs of every length that the repair treats differently, and
keys that must be sorted digit by digit."""
import numpy as np
import pytest

from conftest import log
from oracle import oracle as o
from test_gpu_radix_sort import same_bits, sort_keys, sort_pairs
from test_gpu_small_sort import rank_path  # noqa: F401  (both ranking paths)

pytestmark = pytest.mark.gpu


def layouts(n, rng):
    """name -> n uint64 sort keys"""
    full = rng.integers(0, 1 << 64, n, dtype=np.uint64)
    out = {"uniform": full}
    # groups of equal upper 40 bits: pairs, short runs, runs ranked in LDS (33..2112), longer ones
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
