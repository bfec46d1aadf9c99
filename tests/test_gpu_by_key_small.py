"""ScanByKey and ReduceByKey of small inputs (one launch, every tile finds the
run that enters it by itself): sizes at the edges of its 4096-element tiles and
of its range, runs that span any number of tiles."""
import numpy as np
import pytest

from conftest import log
from oracle import oracle as o

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 4095, 4096, 4097, 8192, 12_289, 65_535, 65_536, 65_537]


def keys_of(dtype, n, run, seed):
    rng = np.random.default_rng(seed)
    k = np.cumsum(rng.random(n) < 1.0 / run).astype(dtype)
    if run == 50_000:
        k[:] = 3  # one run
    if np.dtype(dtype).kind == "f" and n > 100:
        k[10:14] = [0.0, -0.0, np.nan, np.nan]  # equal, equal, never equal
    return k


@pytest.mark.parametrize("kdt,vdt", [(np.int32, np.int32), (np.int64, np.int64), (np.float32, np.int32),
                                     (np.uint32, np.uint64)])
@pytest.mark.parametrize("run", [1, 3, 128, 5000, 50_000])
@pytest.mark.parametrize("pad", [0, 1])
def test_vs_oracle(gpu, kdt, vdt, run, pad):
    import gpu_util as g
    from lc_parallel_primitive_amd import DeviceReduce, DeviceScan

    kn, vn = np.dtype(kdt).name, np.dtype(vdt).name
    for n in SIZES:
        log(f"by key small {kn} {vn} n={n} run={run}")
        k, v = keys_of(kdt, n, run, n), g.random_array(vdt, n, seed=n)
        dk, dv = g.to_dev(k, pad), g.to_dev(v, pad)
        tmp = g.temp(DeviceScan.GetScanByKeyTempStorageBytes(kn, vn, n))
        for op, code in (("sum", o.OP_SUM), ("max", o.OP_MAX)):
            for inclusive in (False, True):
                out = g.empty(n, vdt, pad)
                s = DeviceScan()
                (s.InclusiveScanByKey if inclusive else s.ExclusiveScanByKey)(tmp, dk, dv, out, op, n, 5)
                assert (g.to_host(out) == o.scan_by_key(k, v, inclusive, code, 5)).all()
        rk, rv = o.reduce_by_key(k, v, o.OP_SUM)
        tmp = g.temp(DeviceReduce.GetReduceByKeyTempStorageBytes(kn, vn, n))
        uo, ao, runs = g.empty(n, kdt, pad), g.empty(n, vdt, pad), g.empty(1, np.uint32)
        DeviceReduce().ReduceByKey(tmp, dk, dv, uo, ao, runs, "sum", n)
        assert g.to_host(runs)[0] == rk.size
        assert g.to_host(uo)[:rk.size].tobytes() == rk.tobytes()
        assert (g.to_host(ao)[:rk.size] == rv).all()


@pytest.mark.parametrize("vdt", [np.float32, np.float64])
def test_float_sums(gpu, vdt):
    import gpu_util as g
    from lc_parallel_primitive_amd import DeviceReduce, DeviceScan

    n = 40_000
    k, v = keys_of(np.int32, n, 700, 1), g.random_array(vdt, n, seed=2)
    dk, dv, out = g.to_dev(k), g.to_dev(v), g.empty(n, vdt)
    vn = np.dtype(vdt).name
    tmp = g.temp(DeviceScan.GetScanByKeyTempStorageBytes("int32", vn, n))
    DeviceScan().InclusiveSumByKey(tmp, dk, dv, out, n)
    ref, ab = o.scan_by_key_f64(k, v, True)
    assert (np.abs(g.to_host(out).astype(np.float64) - ref) <= 1e-5 * ab + 1e-30).all()
    tmp = g.temp(DeviceReduce.GetReduceByKeyTempStorageBytes("int32", vn, n))
    uo, ao, runs = g.empty(n, np.int32), g.empty(n, vdt), g.empty(1, np.uint32)
    DeviceReduce().ReduceByKey(tmp, dk, dv, uo, ao, runs, "sum", n)
    rv, rab = o.reduce_by_key_f64(k, v)
    assert g.to_host(runs)[0] == rv.size
    assert (np.abs(g.to_host(ao)[:rv.size].astype(np.float64) - rv) <= 1e-5 * rab + 1e-30).all()


def test_scan_in_place(gpu):
    """An output over the values takes the look-back path."""
    import gpu_util as g
    from lc_parallel_primitive_amd import DeviceScan

    n = 50_000
    k, v = keys_of(np.int32, n, 300, 3), g.random_array(np.int32, n, seed=4)
    dk, dv = g.to_dev(k), g.to_dev(v)
    tmp = g.temp(DeviceScan.GetScanByKeyTempStorageBytes("int32", "int32", n))
    DeviceScan().InclusiveSumByKey(tmp, dk, dv, dv, n)
    assert (g.to_host(dv) == o.scan_by_key(k, v, True)).all()


@pytest.mark.parametrize("kdt,vdt,tile", [(np.int32, np.int32, 8192), (np.int64, np.uint64, 4096)])
@pytest.mark.parametrize("run", [3, 128, 30_000])
@pytest.mark.parametrize("tiles,extra", [(1023, 5), (1024, 0), (1024, 1), (1100, -3)])
def test_reduce_by_key_where_staging_begins(gpu, kdt, vdt, tile, run, tiles, extra):
    """Inputs whose tiles all wait for their place, and one tile more: tiles with few runs stage them."""
    import gpu_util as g
    from lc_parallel_primitive_amd import DeviceReduce

    n = tiles * tile + extra
    kn, vn = np.dtype(kdt).name, np.dtype(vdt).name
    log(f"reduce by key {kn} {vn} n={n} run={run}")
    k, v = keys_of(kdt, n, run, 7), g.random_array(vdt, n, seed=8)
    rk, rv = o.reduce_by_key(k, v, o.OP_SUM)
    tmp = g.temp(DeviceReduce.GetReduceByKeyTempStorageBytes(kn, vn, n))
    uo, ao, runs = g.empty(n, kdt), g.empty(n, vdt), g.empty(1, np.uint32)
    DeviceReduce().ReduceByKey(tmp, g.to_dev(k), g.to_dev(v), uo, ao, runs, "sum", n)
    assert g.to_host(runs)[0] == rk.size
    assert (g.to_host(uo)[:rk.size] == rk).all() and (g.to_host(ao)[:rk.size] == rv).all()


@pytest.mark.parametrize("n", [3000, 40_000, 300_000])
@pytest.mark.parametrize("ahead", [0, 64, 8192])
def test_reduce_by_key_outputs_over_the_inputs(gpu, n, ahead):
    """Outputs that start `ahead` elements into the inputs, long runs: every
    tile has read its elements before a run is stored."""
    import gpu_util as g
    import torch
    from lc_parallel_primitive_amd import DeviceReduce

    k, v = keys_of(np.int32, n, 600, n), g.random_array(np.int32, n, seed=n)
    rk, rv = o.reduce_by_key(k, v, o.OP_SUM)
    assert rk.size <= n // 400  # fits the tiles' slots, and ends before the last key
    bufs = [torch.empty(n + ahead, dtype=torch.int32, device="cuda") for _ in range(2)]
    for b, a in zip(bufs, (k, v)):
        b[:n].copy_(torch.from_numpy(a))
    runs = g.empty(1, np.uint32)
    tmp = g.temp(DeviceReduce.GetReduceByKeyTempStorageBytes("int32", "int32", n))
    log(f"reduce by key over its inputs n={n} ahead={ahead}")
    DeviceReduce().ReduceByKey(tmp, bufs[0][:n], bufs[1][:n], bufs[0][ahead:], bufs[1][ahead:], runs, "sum", n)
    assert g.to_host(runs)[0] == rk.size
    assert (g.to_host(bufs[0])[ahead:ahead + rk.size] == rk).all()
    assert (g.to_host(bufs[1])[ahead:ahead + rk.size] == rv).all()


@pytest.mark.parametrize("kdt,vdt", [(np.int32, np.int32), (np.int64, np.uint64)])
@pytest.mark.parametrize("tiles", [9, 63, 64, 65, 128, 200, 1024, 1025])
def test_reduce_by_key_runs_of_many_tiles(gpu, kdt, vdt, tiles):
    """Tiles inside one run wait for nothing, and every 64th publishes the
    fold up to its end: runs that span from a few tiles to all of them, on
    both sides of the line to staged runs (1024 tiles)."""
    import gpu_util as g
    from lc_parallel_primitive_amd import DeviceReduce

    tile = 32_768 // np.dtype(vdt).itemsize
    kn, vn = np.dtype(kdt).name, np.dtype(vdt).name
    for n in (tiles * tile, tiles * tile - tile + 1):
        v = g.random_array(vdt, n, seed=n)
        dv = g.to_dev(v)
        for heads in ([], [n - 1], [tile * 5], [1, tile * 7 - 1, n // 2, n // 2 + 1], [n // 3]):
            k = np.zeros(n, kdt)
            k[[h for h in heads if h < n]] = 1
            k = np.cumsum(k).astype(kdt)
            log(f"reduce by key {kn} {vn} tiles={tiles} n={n} heads={heads}")
            rk, rv = o.reduce_by_key(k, v, o.OP_SUM)
            tmp = g.temp(DeviceReduce.GetReduceByKeyTempStorageBytes(kn, vn, n))
            uo, ao, runs = g.empty(n, kdt), g.empty(n, vdt), g.empty(1, np.uint32)
            DeviceReduce().ReduceByKey(tmp, g.to_dev(k), dv, uo, ao, runs, "sum", n)
            assert g.to_host(runs)[0] == rk.size
            assert (g.to_host(uo)[:rk.size] == rk).all() and (g.to_host(ao)[:rk.size] == rv).all()
