"""Grouped projections in one GEMM launch (gemm_group_route, gemm.hip): every
route at its row and tile edges, with siblings of unequal, odd and empty
widths, against the single projections (bit for bit) and the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from inferrous_amd import CudaContext, DeviceBuffer, load

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.fixture(scope="module")
def env():
    ctx = CudaContext(0)
    return load(ctx), ctx.new_stream()


def dev(s, a):
    return DeviceBuffer.from_host(s, np.ascontiguousarray(a))


def check(env, m, k, ns, dtype, oracle_rows=2):
    mod, s = env
    print(f"grouped m={m} k={k} n={ns} {np.dtype(dtype).name}", flush=True)
    rng = np.random.default_rng(m * 31 + k + sum(ns))
    q = rng.integers(-127, 128, (m, k), dtype=np.int8)
    asc = (rng.random(m) / 512 + 1e-4).astype(F32)
    dq, da = dev(s, q), dev(s, asc)
    host = [(rng.integers(-127, 128, (n, k), dtype=np.int8), (rng.random(n) / 256).astype(F32)) for n in ns]
    mats = [(dev(s, w), dev(s, sc)) for w, sc in host]
    guard = 64  # values past each output that must stay as they are
    outs = [dev(s, np.full(m * n + guard, 7, dtype)) for n in ns]
    mod.linear_grouped(s, dq, da, k, [(w, sc, DeviceBuffer.view_of(o, 0, m * n))
                                      for (w, sc), o, n in zip(mats, outs, ns)])
    for (w, sc), (hw, hs), o, n in zip(mats, host, outs, ns):
        got = o.to_host_vec(s)
        assert (got[m * n:] == 7).all()
        if n == 0:
            continue
        one = DeviceBuffer.zeroed(s, m * n, dtype)
        mod.linear(s, None, dq, da, w, sc, k, one)
        assert np.array_equal(got[:m * n].view(np.uint8), one.to_host_vec(s).view(np.uint8)), n
        rows = sorted({0, m - 1})[:oracle_rows]
        acc, of, ob = oracle.linear(q[rows], asc[rows], hw, hs, k, threads=8)
        want = {np.int32: acc, np.uint16: ob, np.float32: of}[dtype]
        assert np.array_equal(got[:m * n].reshape(m, n)[rows].ravel().view(np.uint8), want.ravel().view(np.uint8))


@pytest.mark.parametrize("m", [1, 2, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65, 129, 160, 161, 256, 257, 300])
@pytest.mark.parametrize("k,ns", [(512, (200, 33, 1)), (1024, (64, 0, 96, 31)), (8192, (40, 17))])
def test_rows_and_ragged_columns(env, m, k, ns):
    check(env, m, k, ns, np.uint16)


@pytest.mark.parametrize("m", [17, 24, 25, 32, 33, 40, 41, 48, 49, 56, 57, 64])
@pytest.mark.parametrize("k,ns", [(512, (4100, 33, 1, 7)), (4096, (4096, 1024, 1024))])
def test_narrow_two_column_blocks(env, m, k, ns):
    """gemm_narrow on 32 columns per workgroup (and, for the single
    projections, on 16), every count of live activation loads."""
    check(env, m, k, ns, np.uint16)


@pytest.mark.parametrize("m", [3, 16, 40, 130, 250])
@pytest.mark.parametrize("dtype", [np.float32, np.int32])
def test_wide_group_one_m_tile(env, m, dtype):
    """224 and more tiles of 96 columns: the unsplit one-M-tile kernel."""
    check(env, m, 128, (10000, 11600, 5), dtype)


@pytest.mark.parametrize("ns", [(15000, 8100), (8000, 7400, 1), (3000, 3300), (500, 100)])
@pytest.mark.parametrize("dtype", [np.uint16, np.float32, np.int32])
def test_prefill_tiles(env, ns, dtype):
    """256 x 192, 128 x 192, 128 x 128 and 128 x 64 tiles."""
    check(env, 512 if sum(ns) > 6000 else 257, 384, ns, dtype)


@pytest.mark.parametrize("m", [2, 5, 70, 300])
def test_k_without_a_grouped_route(env, m):
    """K % 128 != 0: one launch per matrix, as before."""
    check(env, m, 1040, (100, 33), np.uint16)
