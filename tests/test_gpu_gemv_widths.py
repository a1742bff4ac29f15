"""The M = 1 GEMV with its activation row in registers (gemv_m1_one, gemv_m1)
at every K it takes, on odd row counts, with a residual, for siblings and for
the fused selection, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from inferrous_amd import CudaContext, DeviceBuffer, load
from test_indexing import argmax_route, check_gemv_m1, route

F32 = np.float32


@pytest.mark.parametrize("kc", range(1, 18))
def test_routes(kc):
    for n in (1, 3, 4097, 9001):
        r = route(1, n, kc * 1024)
        assert r["family"] == (1 if kc <= 16 else 3)
        if kc <= 16:
            check_gemv_m1(1, n, kc * 1024, r, False)
        a = argmax_route(n, kc * 1024)
        assert a["family"] == (2 if kc <= 12 else 3)
        if kc <= 12:
            check_gemv_m1(1, n, kc * 1024, a, False, argmax=True)


@pytest.mark.gpu
@pytest.mark.parametrize("kc", range(1, 18))
@pytest.mark.parametrize("n", [1, 7, 1003])
def test_every_width(kc, n):
    ctx = CudaContext(0)
    mod, s = load(ctx), ctx.new_stream()
    k = kc * 1024
    rng = np.random.default_rng(k + n)
    dev = lambda a: DeviceBuffer.from_host(s, np.ascontiguousarray(a))  # noqa: E731
    q, asc = rng.integers(-127, 128, (1, k), dtype=np.int8), np.array([0.01], F32)
    host = [(rng.integers(-127, 128, (m, k), dtype=np.int8), (rng.random(m) / 99).astype(F32)) for m in (n, 5)]
    res = oracle.bf16_rne(rng.standard_normal(n).astype(F32))
    want = [oracle.linear(q, asc, w, ws, k) for w, ws in host]
    dq, da, mats = dev(q), dev(asc), [(dev(w), dev(ws)) for w, ws in host]
    out, comb, tok = DeviceBuffer.zeroed(s, n, F32), DeviceBuffer.zeroed(s, n, F32), DeviceBuffer.zeroed(s, 1, np.uint32)
    mod.linear_residual(s, None, dq, da, *mats[0], k, dev(res), out, comb)
    assert np.array_equal(out.to_host_vec(s), want[0][1].ravel())
    assert np.array_equal(comb.to_host_vec(s), oracle.residual(res, want[0][1].ravel()))
    outs = [DeviceBuffer.zeroed(s, m, np.uint16) for m in (n, 5)]
    mod.linear_pair(s, None, dq, da, k, *mats[0], outs[0], *mats[1], outs[1])
    for o, w in zip(outs, want):
        assert np.array_equal(o.to_host_vec(s), w[2].ravel())
    mod.linear_argmax(s, dq, da, *mats[0], k, tok, out)
    assert np.array_equal(out.to_host_vec(s), want[0][1].ravel())
    assert int(tok.to_host_vec(s)[0]) == oracle.argmax(want[0][1].ravel())
