"""gemm_dma's tiles: the strip numbering and the bounds of the 32-bit lane
offsets on the CPU, and every tile with whole, ragged and several strips of M
tiles on the GPU, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from test_indexing import route, xcd_slot

STRIP, MAX_K, MAX_COLS = 4, 1 << 23, 1 << 26  # kStrip, kMaxK, kMaxCols (gemm.hip)


@pytest.mark.parametrize("tm", [1, 2, 3, 4, 5, 7, 8, 9, 16, 33])
@pytest.mark.parametrize("tn", [1, 2, 16, 31])
@pytest.mark.parametrize("splits", [1, 2])
def test_strip_numbering_visits_every_tile_once(tm, tn, splits):
    T = tm * tn
    L = xcd_slot(np.arange(T * splits), T * splits)
    split, t = L // T, L % T
    strip = STRIP * tn
    s0, inside = t // strip * STRIP, t % strip
    sm = np.minimum(STRIP, tm - s0)
    mt, nt = s0 + inside % sm, inside // sm
    assert mt.max() < tm and nt.max() < tn
    assert len({*zip(split.tolist(), mt.tolist(), nt.tolist())}) == T * splits


def test_lane_offsets_fit_32_bits():
    """The routes that hold a lane's offset in 32 bits stop where it would not
    fit, and the others take over."""
    assert 255 * MAX_K + 127 < 1 << 32               # a tile's last row and chunk, in bytes
    assert (4 * MAX_COLS + 31) * 4 < 1 << 32         # four rows and 31 columns of f32
    for m in (1, 16, 40, 64, 100, 300, 5000):
        for n, k, staged in ((1000, MAX_K, True), (1000, MAX_K + 128, False), (MAX_COLS, 128, True),
                             (MAX_COLS + 4, 128, False)):
            if m * n >= 1 << 32:
                continue
            fam = route(m, n, k, path=2)["family"]
            # unstaged: 64-bit row pointers (gemm_skinny, gemm_narrow, the four-wave tiles with a K tail)
            assert staged or fam in ((11, 15) if m <= 16 else (14,)), (m, n, k, fam)


# (tile, family, m, n, k): eight waves (13), four waves (14), K tails of 16 and
# 112 bytes, K below one stage
TILES = [((128, 64), 13, 2049, 515, 1280), ((128, 128), 13, 1025, 2003, 1280), ((128, 192), 13, 1300, 3003, 1280),
         ((256, 128), 13, 1025, 6003, 1280), ((256, 192), 13, 1300, 6003, 1280), ((64, 128), 13, 129, 10003, 1280),
         ((256, 256), 13, 2049, 6003, 1280), ((64, 64), 14, 150, 515, 1280), ((64, 64), 14, 65, 33, 16),
         ((64, 64), 14, 77, 1003, 112), ((64, 64), 14, 257, 515, 1392), ((128, 64), 14, 1025, 2003, 16),
         ((128, 128), 14, 1300, 3003, 144), ((256, 128), 14, 2049, 2003, 1296), ((256, 256), 14, 1300, 6003, 1296)]


@pytest.mark.parametrize("tile,family,m,n,k", TILES)
def test_tile_routes(tile, family, m, n, k):
    r = route(m, n, k)
    assert (r["family"], r["bm"], r["bn"]) == (family, *tile)


@pytest.mark.parametrize("m,n,k,tile", [(300, 4096, 4096, (128, 64)), (700, 2560, 8192, (128, 64)),
                                        (400, 3584, 8192, (128, 64)), (129, 6144, 4096, (128, 64)),
                                        (180, 6144, 4096, (128, 64)), (129, 8192, 4096, (64, 128)),
                                        (129, 10240, 4096, (64, 128)), (320, 6144, 4096, (64, 128))])
def test_measured_tile_choice(m, n, k, tile):
    """Between the two tiles of 8192 outputs: the one that was faster with
    distinct weights (128 x 64 but where it needs more tiles)."""
    r = route(m, n, k)
    assert (r["bm"], r["bn"]) == tile


@pytest.mark.parametrize("tile,family,m,n,k", [c for c in TILES if c[4] % 128])
def test_tail_reads_stay_inside(tile, family, m, n, k):
    """gemm_dma's DMA sources with a partial last stage (loadA, loadB): every
    16-byte read of every tile lies inside its operand, each live row's chunks
    below K are read once, and a chunk past K meets zeros."""
    bm, bn = tile
    stages = k // 128 + 1
    for rows, b in ((m, bm), (n, bn)):
        row, c = np.divmod(np.arange(b * 8), 8)
        chunk = (c ^ ((row >> 1) & 7)) * 16
        kk = np.arange(stages)[:, None] * 128 + chunk
        for first in range(0, rows, b):
            src = np.where(first + row < rows, row, 0)
            live = kk < k
            at = (first + src) * k + np.where(live, kk, 0)  # weights; activations past K read zeros instead
            assert at.min() >= 0 and (at + 16).max() <= rows * k
            for r in {0, min(b, rows - first) - 1}:
                assert np.array_equal(np.sort(kk[:, row == r][live[:, row == r]]), np.arange(0, k, 16))


@pytest.mark.gpu
@pytest.mark.parametrize("tile,family,m,n,k", TILES)
def test_every_tile(tile, family, m, n, k):
    """Odd M and N (guarded edges beside whole tiles), every output form,
    guard values past the output untouched."""
    from inferrous_amd import CudaContext, DeviceBuffer, load
    ctx = CudaContext(0)
    mod, s = load(ctx), ctx.new_stream()
    print(f"tile {tile} m={m} n={n} k={k}", flush=True)
    rng = np.random.default_rng(m + n)
    q = rng.integers(-127, 128, (m, k), dtype=np.int8)
    w = rng.integers(-127, 128, (n, k), dtype=np.int8)
    asc, ws = (rng.random(m) / 64).astype(np.float32), (rng.random(n) / 64).astype(np.float32)
    res = oracle.bf16_rne(rng.standard_normal(m * n).astype(np.float32))
    acc, of, ob = oracle.linear(q, asc, w, ws, k, threads=8)
    comb = oracle.residual(res, of)
    dev = lambda a: DeviceBuffer.from_host(s, np.ascontiguousarray(a))  # noqa: E731
    dq, da, dw, dws, dres = dev(q), dev(asc), dev(w), dev(ws), dev(res)
    guard = 512
    for dtype, residual in ((np.int32, False), (np.float32, False), (np.uint16, False), (np.float32, True),
                            (np.uint16, True)):
        bufs = [dev(np.full(m * n + guard, 7, dtype)) for _ in range(1 + residual)]
        out, *cb = [DeviceBuffer.view_of(b, 0, m * n) for b in bufs]
        if residual:
            mod.linear_residual(s, None, dq, da, dw, dws, k, dres, out, cb[0])
        else:
            mod.linear_mfma(s, None, dq, da, dw, dws, k, out)
        want = [{np.int32: acc, np.float32: of, np.uint16: ob}[dtype]]
        if residual:
            want.append(comb if dtype == np.float32 else (comb.view(np.uint32) >> 16).astype(np.uint16))
        for b, v in zip(bufs, want):
            got = b.to_host_vec(s)
            assert np.array_equal(got[:m * n].view(np.uint8), v.reshape(-1).view(np.uint8)), (dtype, residual)
            assert (got[m * n:] == 7).all(), (dtype, residual)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(512, 6003, 128), (512, 6003, 1280), (768, 4003, 1280), (769, 4003, 1280),
                                   (5000, 60, 1280), (22000, 60, 640), (33000, 61, 256), (300, 2003, 16384)])
def test_rotated_k(m, n, k):
    """Both sides of gemm_dma's rule for starting each tile at its own K stage
    (one round of tiles in one column): the sums."""
    from inferrous_amd import CudaContext, DeviceBuffer, load
    ctx = CudaContext(0)
    mod, s = load(ctx), ctx.new_stream()
    print(f"rotated m={m} n={n} k={k}", flush=True)
    rng = np.random.default_rng(m + n)
    q = rng.integers(-127, 128, (m, k), dtype=np.int8)
    w = rng.integers(-127, 128, (n, k), dtype=np.int8)
    asc, ws = np.ones(m, np.float32), np.ones(n, np.float32)
    acc, _, _ = oracle.linear(q, asc, w, ws, k, threads=8)
    dq, da, dw, dws = (DeviceBuffer.from_host(s, np.ascontiguousarray(a)) for a in (q, asc, w, ws))
    out = DeviceBuffer.zeroed(s, m * n, np.int32)
    mod.linear(s, None, dq, da, dw, dws, k, out)
    assert np.array_equal(out.to_host_vec(s), acc.reshape(-1))
