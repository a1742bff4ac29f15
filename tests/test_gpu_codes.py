"""Quantizer codes without a division per value (code_bits,
device_common.hpp): the correctly rounded quotient's code at values a few
ulps either side of every rounding boundary, for scales over the whole range,
NaN with payloads and infinities, against the oracle's division."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from inferrous_amd import CudaContext, DeviceBuffer, load

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module")
def env():
    ctx = CudaContext(0)
    return load(ctx), ctx.new_stream()


def boundary_rows(rng, rows, width, bf16):
    """Row r: its maximum m, then (k + 0.5) s for s = RN(m / 127), moved by up
    to three representable steps; bf16: every value a BF16 one."""
    m = np.exp(rng.uniform(-18, 80, rows)).astype(F)
    if bf16:
        m = oracle.bf16_rne(m)
    s = (m / F(127)).astype(F)
    x = ((rng.integers(-127, 127, (rows, width)).astype(F) + F(0.5)) * s[:, None]).astype(F)
    u = x.view(np.uint32).copy()
    step = rng.integers(-3, 4, u.shape)
    if bf16:
        u = ((u >> 16).astype(np.int64) + step).astype(np.uint32) << 16
    else:
        u = (u.astype(np.int64) + step).astype(np.uint32)
    x = np.clip(u.view(F), -m[:, None], m[:, None]).astype(F)
    x[:, 7] = m
    x[0, 9:12] = np.array([0x7FC00001, 0xFFC12345, 0x7F800000], np.uint32).view(F)  # NaNs, then an infinite scale
    x[1, 9:12] = np.array([0x7FC000FF, 0xFFFFFFFF, 0x7F8000FF], np.uint32).view(F)  # NaNs only
    x[2] = 0.0
    return x


@pytest.mark.parametrize("width", [256, 1000, 1001, 4096, 5120, 12288, 16384, 16400])
@pytest.mark.parametrize("bf16", [False, True])
def test_codes_at_rounding_boundaries(env, width, bf16):
    mod, s = env
    rng = np.random.default_rng(width + bf16)
    rows = 48
    x = boundary_rows(rng, rows, width, bf16)
    if bf16:
        xb = (x.reshape(-1).view(np.uint32) >> 16).astype(np.uint16)
        want_q, want_s = oracle.quantize_bf16(xb, width)
        x = xb
    else:
        x = x.reshape(-1)
        want_q, want_s = oracle.quantize(x, width)
    q, sc = DeviceBuffer.zeroed(s, rows * width, np.int8), DeviceBuffer.zeroed(s, rows, F)
    mod.quantize(s, None, DeviceBuffer.from_host(s, x), width, q, sc)
    assert np.array_equal(sc.to_host_vec(s).view(np.uint32), want_s.view(np.uint32))
    assert np.array_equal(q.to_host_vec(s), want_q)


def test_norm_codes(env):
    """norm_quantize's codes are those of its own output rows, also for rows
    holding NaN, infinities and zeros."""
    mod, s = env
    rng = np.random.default_rng(3)
    rows = 200
    x = (rng.standard_normal((rows, 4096)) * np.exp(rng.uniform(-20, 20, (rows, 1)))).astype(F)
    x[0, 3] = np.nan
    x[1, 5] = np.inf
    x[2] = 0.0
    gain = (1 + 0.1 * rng.standard_normal(4096)).astype(F)
    out, q = DeviceBuffer.zeroed(s, rows * 4096, F), DeviceBuffer.zeroed(s, rows * 4096, np.int8)
    sc, mx = DeviceBuffer.zeroed(s, rows, F), DeviceBuffer.zeroed(s, rows, np.uint32)
    mod.norm_quantize(s, None, DeviceBuffer.from_host(s, x.reshape(-1)), DeviceBuffer.from_host(s, gain), out, q, sc, mx)
    want_q, want_s = oracle.quantize(out.to_host_vec(s), 4096)
    assert np.array_equal(q.to_host_vec(s), want_q)
    assert np.array_equal(sc.to_host_vec(s).view(np.uint32), want_s.view(np.uint32))
