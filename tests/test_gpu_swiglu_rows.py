"""The one-pass SwiGLU rows (swiglu_rows, gemv.hip) at the edges of its
vectors, its register-held width and its alignment rule: act equal to the
elementwise form bit for bit and within one BF16 ulp of the oracle, the
maxima equal to the fold of what was written, and the codes equal to
quantize_with_max of act with the folded maxima."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from inferrous_amd import CudaContext, DeviceBuffer, load
from inferrous_amd._lib import OUT_BF16, OUT_F32, lib
from test_gpu_swiglu import F32, FLOOR, act_close, bits, dev, fold_max

pytestmark = pytest.mark.gpu

INF, NAN = np.inf, np.nan


@pytest.fixture(scope="module")
def env():
    ctx = CudaContext(0)
    return load(ctx), ctx.new_stream()


def values(buf, s):
    a = buf.to_host_vec(s)
    return a if a.dtype == F32 else (a.astype(np.uint32) << 16).view(F32)


@pytest.mark.parametrize("width", [1, 7, 8, 2048, 2056, 4096, 4100, 8200, 12288, 16384, 16385, 16392])
@pytest.mark.parametrize("dtype", [np.float32, np.uint16])
@pytest.mark.parametrize("shift", [0, 1])
def test_rows_equal_the_elementwise_form(env, width, dtype, shift):
    mod, s = env
    rows = 5
    rng = np.random.default_rng(width + shift)
    g, u = (oracle.bf16_rne((rng.standard_normal(rows * width) * 3).astype(F32)) for _ in range(2))
    g[:4], u[:4] = [NAN, INF, -INF, 0.0][:len(g[:4])], 1.0
    u[-1] = INF
    enc = (lambda a: a) if dtype == np.float32 else (lambda a: (bits(a) >> 16).astype(np.uint16))

    def shifted(a):
        """The array `shift` elements past a 16-byte boundary."""
        whole = dev(s, np.concatenate([np.zeros(shift, dtype), a]))
        return DeviceBuffer.view_of(whole, shift, len(a))

    dg, du = shifted(enc(g)), shifted(enc(u))
    flat, act = (shifted(np.zeros(rows * width, dtype)) for _ in range(2))
    start = np.full(rows, FLOOR, np.uint32)
    start[1] = bits(F32(1e30))[0]
    mx = dev(s, start)
    code = OUT_F32 if dtype == np.float32 else OUT_BF16
    assert lib().w8a8_swiglu(s.handle, dg.ptr, du.ptr, rows, width, flat.ptr, None, code) == 0
    assert lib().w8a8_swiglu(s.handle, dg.ptr, du.ptr, rows, width, act.ptr, mx.ptr, code) == 0
    got, want = values(act, s).reshape(rows, width), values(flat, s).reshape(rows, width)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    fin = np.isfinite(got.ravel())
    act_close(got.ravel()[fin], g[fin], u[fin])
    maxima = mx.to_host_vec(s)
    for r in range(rows):
        assert int(maxima[r]) == max(int(start[r]), fold_max(got[r])), f"row {r}"
    # in place: act over gate
    assert lib().w8a8_swiglu(s.handle, dg.ptr, du.ptr, rows, width, dg.ptr, dev(s, start).ptr, code) == 0
    assert np.array_equal(values(dg, s).view(np.uint32), got.ravel().view(np.uint32))


@pytest.mark.parametrize("n", [7, 8, 2048, 4100, 16384, 16385])
@pytest.mark.parametrize("dtype", [np.float32, np.uint16])
@pytest.mark.parametrize("m", [6, 70])
def test_row_codes(env, m, n, dtype):
    """linear_swiglu_quantize at several rows: the codes and scales of act
    under the folded maxima, one row's maximum set beforehand to a larger and
    one to a smaller value than its own."""
    mod, s = env
    k = 32
    rng = np.random.default_rng(m + n)
    mats = [(dev(s, rng.integers(-127, 128, (n, k), dtype=np.int8)), dev(s, (rng.random(n) / 64).astype(F32)))
            for _ in range(2)]
    q, asc = dev(s, rng.integers(-127, 128, (m, k), dtype=np.int8)), dev(s, (rng.random(m) / 64).astype(F32))
    g, u, act = (DeviceBuffer.zeroed(s, m * n, dtype) for _ in range(3))
    start = np.full(m, FLOOR, np.uint32)
    start[1] = bits(F32(1e6))[0]
    mx = dev(s, start)
    codes, sc = DeviceBuffer.zeroed(s, m * n, np.int8), DeviceBuffer.zeroed(s, m, F32)
    mod.linear_swiglu_quantize(s, None, q, asc, k, *mats[0], g, *mats[1], u, act, mx, codes, sc)
    a = values(act, s)
    act_close(a, values(g, s), values(u, s))
    want = [max(int(start[r]), fold_max(a.reshape(m, n)[r])) for r in range(m)]
    assert mx.to_host_vec(s).tolist() == want
    wq, ws = oracle.quantize_with_max(a, n, np.array(want, np.uint32))
    assert np.array_equal(codes.to_host_vec(s), wq)
    assert np.array_equal(bits(sc.to_host_vec(s)), bits(ws))


@pytest.mark.parametrize("n", [7, 2048])
@pytest.mark.parametrize("dtype", [np.float32, np.uint16])
def test_row_codes_under_a_nan_maximum(env, n, dtype):
    """A maximum whose bits are a NaN (the caller's: no producer folds one)
    gives a NaN scale and the codes 0, as quantize_with_max does, whatever
    the payload."""
    mod, s = env
    m, k = 5, 32
    rng = np.random.default_rng(n)
    mats = [(dev(s, rng.integers(-127, 128, (n, k), dtype=np.int8)), dev(s, (rng.random(n) / 64).astype(F32)))
            for _ in range(2)]
    q, asc = dev(s, rng.integers(-127, 128, (m, k), dtype=np.int8)), dev(s, (rng.random(m) / 64).astype(F32))
    g, u, act = (DeviceBuffer.zeroed(s, m * n, dtype) for _ in range(3))
    start = np.array([0x7f800055, 0x7fc00001, 0xffffffff, 0x7fabcdef, FLOOR], np.uint32)
    mx = dev(s, start)
    codes, sc = dev(s, np.full(m * n, 9, np.int8)), DeviceBuffer.zeroed(s, m, F32)
    mod.linear_swiglu_quantize(s, None, q, asc, k, *mats[0], g, *mats[1], u, act, mx, codes, sc)
    a = values(act, s)
    got, scales = codes.to_host_vec(s).reshape(m, n), sc.to_host_vec(s)
    assert np.isnan(scales[:4]).all() and (got[:4] == 0).all()
    assert mx.to_host_vec(s)[:4].tolist() == start[:4].tolist()
    wq, _ = oracle.quantize_with_max(a[4 * n:], n, np.array([fold_max(a[4 * n:])], np.uint32))
    assert np.array_equal(got[4], wq)


@pytest.mark.parametrize("n", [8, 2048, 16400])
@pytest.mark.parametrize("dtype", [np.float32, np.uint16])
@pytest.mark.parametrize("reuse", ["gate", "up"])
def test_codes_over_gate_or_up(env, n, dtype, reuse):
    """The codes and scales may take the memory of gate or up, which nothing
    reads once act exists (rows that other workgroups have not read yet
    included)."""
    mod, s = env
    m, k = 70, 32
    rng = np.random.default_rng(n)
    mats = [(dev(s, rng.integers(-127, 128, (n, k), dtype=np.int8)), dev(s, (rng.random(n) / 64).astype(F32)))
            for _ in range(2)]
    q, asc = dev(s, rng.integers(-127, 128, (m, k), dtype=np.int8)), dev(s, (rng.random(m) / 64).astype(F32))
    size = m * n * np.dtype(dtype).itemsize
    whole = DeviceBuffer.zeroed(s, size + 4 * m, np.int8)
    shared = DeviceBuffer.view_of(whole, 0, m * n, dtype)
    other, act = (DeviceBuffer.zeroed(s, m * n, dtype) for _ in range(2))
    g, u = (shared, other) if reuse == "gate" else (other, shared)
    codes = DeviceBuffer.view_of(whole, size - m * n, m * n)  # the buffer's last bytes: the last rows' inputs
    sc = DeviceBuffer.view_of(whole, 0, m, np.float32) if dtype == np.float32 else DeviceBuffer.zeroed(s, m, F32)
    mx = dev(s, np.full(m, FLOOR, np.uint32))
    mod.linear_swiglu_quantize(s, None, q, asc, k, *mats[0], g, *mats[1], u, act, mx, codes, sc)
    a = values(act, s)
    plain = [DeviceBuffer.zeroed(s, m * n, dtype) for _ in range(3)]
    mod.linear_swiglu(s, None, q, asc, k, *mats[0], plain[0], *mats[1], plain[1], plain[2], None)
    assert np.array_equal(a.view(np.uint32), values(plain[2], s).view(np.uint32))
    want = [fold_max(row) for row in a.reshape(m, n)]
    assert mx.to_host_vec(s).tolist() == want
    wq, ws = oracle.quantize_with_max(a, n, np.array(want, np.uint32))
    assert np.array_equal(codes.to_host_vec(s), wq)
    assert np.array_equal(bits(sc.to_host_vec(s)), bits(ws))


@pytest.mark.parametrize("rows,width", [(1, 16384), (4, 12288), (5, 12288), (300, 512), (300, 513), (8, 1024),
                                        (8, 1025), (32, 256), (70000, 3)])
@pytest.mark.parametrize("dtype", [np.float32, np.uint16])
def test_route_edges_without_codes(env, rows, width, dtype):
    """Either side of the lines between swiglu_kernel and swiglu_rows (and
    more rows than a grid's y extent): act and the folded maxima."""
    mod, s = env
    rng = np.random.default_rng(rows + width)
    g, u = (oracle.bf16_rne((rng.standard_normal(rows * width) * 3).astype(F32)) for _ in range(2))
    enc = (lambda a: a) if dtype == np.float32 else (lambda a: (bits(a) >> 16).astype(np.uint16))
    dg, du = dev(s, enc(g)), dev(s, enc(u))
    flat, act = (DeviceBuffer.zeroed(s, rows * width, dtype) for _ in range(2))
    start = np.full(rows, FLOOR, np.uint32)
    start[rows // 2] = bits(F32(1e30))[0]
    mx = dev(s, start)
    code = OUT_F32 if dtype == np.float32 else OUT_BF16
    assert lib().w8a8_swiglu(s.handle, dg.ptr, du.ptr, rows, width, flat.ptr, None, code) == 0
    assert lib().w8a8_swiglu(s.handle, dg.ptr, du.ptr, rows, width, act.ptr, mx.ptr, code) == 0
    got = values(act, s).reshape(rows, width)
    assert np.array_equal(got.view(np.uint32), values(flat, s).reshape(rows, width).view(np.uint32))
    act_close(got.ravel(), g, u)
    assert np.array_equal(mx.to_host_vec(s), np.maximum(start, (got.view(np.uint32) & 0x7fffffff).max(axis=1)))
