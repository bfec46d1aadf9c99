"""The one-workgroup sort of small inputs: the sizes at which the items per
thread and the path change, on both ranking paths, with outputs that alias the
inputs."""
import numpy as np
import pytest

from conftest import log
from oracle import oracle as o
from test_gpu_radix_sort import same_bits, sort_keys, sort_pairs

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[1, 2], ids=["atomic", "match"])
def rank_path(gpu, request):
    import lc_parallel_primitive_amd as lcpp

    L = lcpp.lib()
    assert L.lcpp_test_set_sort_rank_path(request.param) == 0
    yield
    assert L.lcpp_test_set_sort_rank_path(0) == 0


def keys_of(dtype, n, seed):
    """Full-range keys with a run of equal ones, -0.0 and +0.0, and infinities among them."""
    import gpu_util as g

    a = g.random_array(dtype, n, seed=seed)
    a[n // 3:n // 2] = a[n // 3] if n > 1 else a[0]
    if a.dtype.kind == "f" and n > 8:
        a[1::7], a[2::11], a[3], a[4] = -0.0, 0.0, np.inf, -np.inf
    return a


@pytest.mark.parametrize("kdt,vdt", [(np.uint32, np.float32), (np.float32, np.int64), (np.uint64, np.uint32),
                                     (np.float64, np.float64)])
@pytest.mark.parametrize("n", [1, 2, 64, 1025, 2047, 2048, 2049, 8191, 8192, 8193, 16383, 16384, 16385])
@pytest.mark.parametrize("descending", [False, True])
def test_edges_vs_oracle(rank_path, kdt, vdt, n, descending):
    import gpu_util as g

    k = keys_of(kdt, n, n)
    v = g.random_array(vdt, n, seed=n + 1)
    log(f"small sort {np.dtype(kdt).name} {np.dtype(vdt).name} n={n} desc={descending}")
    rk, rv = o.radix_sort(k, v, descending=descending)
    dk, dv = g.to_dev(k), g.to_dev(v)
    ko, vo = sort_pairs(dk, dv, n, kdt, vdt, descending)
    assert same_bits(g.to_host(ko), rk) and same_bits(g.to_host(vo), rv)
    assert same_bits(g.to_host(dk), k) and same_bits(g.to_host(dv), v)  # inputs preserved
    assert same_bits(g.to_host(sort_keys(g.to_dev(k, 1), n, kdt, pad=1, descending=descending)), rk)


@pytest.mark.parametrize("n", [2048, 8192])
def test_outputs_may_alias_inputs(rank_path, n):
    import gpu_util as g
    from lc_parallel_primitive_amd import DeviceRadixSort

    k = keys_of(np.uint32, n, 5)
    v = g.random_array(np.uint64, n, seed=6)
    dk, dv = g.to_dev(k), g.to_dev(v)
    tmp = g.temp(DeviceRadixSort.GetSortPairsTempStorageBytes("uint32", "uint64", n))
    DeviceRadixSort().SortPairs(tmp, dk, dk, dv, dv, n)
    rk, rv = o.radix_sort(k, v)
    assert same_bits(g.to_host(dk), rk) and same_bits(g.to_host(dv), rv)


@pytest.mark.parametrize("kdt,vdt", [(np.uint32, None), (np.float32, None), (np.uint64, None), (np.float32, np.uint32),
                                     (np.int32, np.int64), (np.float64, np.uint32)])
@pytest.mark.parametrize("n", [(1 << 19) - 1, 1 << 19, (1 << 19) + 1, 3 << 19, (3 << 19) + 4095, 1 << 21,
                               (1 << 21) + 2, 1 << 22, (1 << 22) + 1])
def test_tile_sizes_change(rank_path, kdt, vdt, n):
    """Keys with one frequent value (a hot digit in every pass) on either side of every line at which the
    tiles change, and temp storage that a smaller sort always fits."""
    import gpu_util as g
    from lc_parallel_primitive_amd import DeviceRadixSort

    k = g.random_array(kdt, n, seed=n % 1000)
    k[::5] = k[0]
    log(f"sort {np.dtype(kdt).name} {vdt} n={n}")
    if vdt is None:
        name = np.dtype(kdt).name
        sizes = [DeviceRadixSort.GetSortKeysTempStorageBytes(name, m) for m in (n - 4097, n - 1, n)]
        assert sizes == sorted(sizes)
        assert same_bits(g.to_host(sort_keys(g.to_dev(k), n, kdt)), o.radix_sort(k, nthreads=8))
    else:
        v = g.random_array(vdt, n, seed=1)
        rk, rv = o.radix_sort(k, v, nthreads=8)
        ko, vo = sort_pairs(g.to_dev(k), g.to_dev(v), n, kdt, vdt)
        assert same_bits(g.to_host(ko), rk) and same_bits(g.to_host(vo), rv)
