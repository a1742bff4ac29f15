"""The indexing contract of every kernel route, checked on the CPU.

For each projection shape the library's own host routing decides the
launch (w8a8_diag_linear_route / w8a8_diag_argmax_route: the kernel family,
its compile-time shape and grid -- gemm_route / gemv_route in the library),
and this file replays that kernel's address arithmetic over the whole grid,
with numpy over every workgroup, wave and lane.  Every global read must lie
inside its operand, every LDS access inside the kernel's LDS array, every
store inside its output, and every output element (every slab element for a
split-K launch) must be written exactly once.  K loops are checked at their
extreme iterations: each address is affine in the loop counter.

The replay restates the index expressions of the kernels, each function
naming the kernel it follows; the table in the design notes states the
same bounds in words.  Shapes: the benchmark configurations (C1-C5: the
decode shapes at M = 1, the lm_head, M = 129 and 512, the ragged M = 4 / 16 /
64), the M = 129 tails (M = 129-135 and 136-159, sampled), N not a multiple
of 96, K not a multiple of 128, and the folded producers' and SwiGLU
kernels' fixed launch shapes.  This is the reference's checked build
(tools/cuda.sh:15-19) in host form.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from conftest import seeded_linear_shapes
from inferrous_amd import _lib

F32, BF16, I32 = 0, 1, 2  # W8A8_OUT_* (include/inferrous_w8a8.h)
AUTO, DOT4, MFMA = 0, 1, 2  # W8A8_PATH_*
ROUTE_LEN = 20
DECODE = [(6144, 4096), (4096, 4096), (24576, 4096), (4096, 12288)]


def route(m, n, k, dtype=BF16, residual=False, path=AUTO, workspace=0):
    r = np.zeros(ROUTE_LEN, np.int32)
    st = _lib.lib().w8a8_diag_linear_route(m, n, k, dtype, int(residual), path, workspace, r.ctypes.data,
                                           ROUTE_LEN)
    assert st == 0, st
    keys = ("family grid_x grid_y block bm bn wm wn sa sb ma mt s u splits nt epi_cols rows kc waves").split()
    return dict(zip(keys, (int(v) for v in r)))


def argmax_route(n, k):
    r = np.zeros(ROUTE_LEN, np.int32)
    assert _lib.lib().w8a8_diag_argmax_route(n, k, r.ctypes.data, ROUTE_LEN) == 0
    keys = ("family grid_x grid_y block bm bn wm wn sa sb ma mt s u splits nt epi_cols rows kc waves").split()
    return dict(zip(keys, (int(v) for v in r)))


def workspace_bytes(m, n, k):
    return int(_lib.lib().w8a8_linear_workspace_bytes(m, n, k))


# ------------------------------------------------------------------ helpers
def within(name, lo, hi, size):
    """Every access [lo, hi) (arrays of byte or element offsets) inside [0, size)."""
    lo = np.asarray(lo)
    hi = np.asarray(hi)
    if lo.size == 0:
        return
    assert lo.min() >= 0, f"{name}: access below the buffer ({lo.min()})"
    assert hi.max() <= size, f"{name}: access past the buffer ({hi.max()} > {size})"


def written_once(name, idx, total):
    """Stores at element offsets idx: inside [0, total) and each element once."""
    idx = np.asarray(idx, np.int64).ravel()
    assert idx.size == total, f"{name}: {idx.size} stores for {total} elements"
    within(name, idx, idx + 1, total)
    counts = np.bincount(idx, minlength=total)
    assert counts.max() == 1 and counts.min() == 1, f"{name}: an element is written {counts.max()} times " \
                                                    f"or not at all"


def xcd_slot(b, G):
    """Workgroup b's slot among G (gemm.hip / gemv.hip xcd_slot): XCD-major when G % 8 == 0."""
    b = np.asarray(b)
    return (b % 8) * (G // 8) + b // 8 if G % 8 == 0 else b


def mfma32_rows_cols(lane, v):
    """Row / column of value v of lane l in a 32 x 32 i32 MFMA block (gemm.hip)."""
    return (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3), lane & 31


def frag_offsets():
    """gemm_dma / gemm_tall fragment reads: lane l, sub-step i -> byte offset
    inside a 32-row block of 128-byte LDS rows (gemm.hip)."""
    lane = np.arange(64)
    fr, fh = lane & 31, lane >> 5
    return np.stack([fr * 128 + (((2 * i + fh) ^ ((fr >> 1) & 7)) * 16) for i in range(4)])  # [4, 64]


# ------------------------------------------------------------------ GEMM routes
def store_blocks(m, n, row0, col0, FM, FN):
    """(rows, cols) that store_blocks writes for wave tiles with top-left
    corners (row0, col0) (broadcast arrays), guarded by r < m, c < n
    (gemm.hip).  Its epilogue loads are clamped (min(r, m - 1),
    min(c, n - 1)), hence always in bounds."""
    lane = np.arange(64)[:, None]
    v = np.arange(16)[None, :]
    rr, cc = mfma32_rows_cols(lane, v)                      # [64, 16]
    # [..., FM, FN, lane, v]
    rows = np.asarray(row0)[..., None, None, None, None] + 32 * np.arange(FM)[:, None, None, None] + rr
    cols = (np.asarray(col0)[..., None, None, None, None] + 32 * np.arange(FN)[:, None, None]
            + np.zeros_like(v) + (lane & 31))
    rows, cols = np.broadcast_arrays(rows, cols)
    keep = (rows < m) & (cols < n)
    return rows[keep].astype(np.int64), cols[keep].astype(np.int64)


STRIP, CUS = 4, 256                    # kStrip, kCus (gemm.hip)
MAX_K, MAX_COLS = 1 << 23, 1 << 26     # kMaxK, kMaxCols
KERNEL_TILES = {13: 8, 14: 4}          # waves per workgroup of gemm_dma's families


def own_tile(ns, bn):
    """Column tiles of the matrices ns (one for a single projection): per tile
    the matrix that own_tile (gemm.hip) picks and the tile's index within it,
    by the kernel's comparisons against the launcher's tbegin."""
    tbegin = np.concatenate([[0], np.cumsum([-(-n // bn) for n in ns])])
    tbegin = np.concatenate([tbegin, np.full(5 - len(tbegin), tbegin[-1])])  # kMaxGroup + 1 entries
    t = np.arange(tbegin[-1])
    mat, first = np.zeros_like(t), np.zeros_like(t)
    for i in range(1, 4):
        mat = np.where(t >= tbegin[i], i, mat)
        first = np.where(t >= tbegin[i], tbegin[i], first)
    return mat, t - first


def check_dma(m, ns, k, r, residual):
    """gemm_dma over its grid, eight waves (family 13) or four (14), with or
    without a K tail, one matrix or several: the strip numbering, the DMA
    sources of every stage, the LDS ring slots, the rotated K order, the
    fragment reads, the stores of store_blocks."""
    ns = [ns] if isinstance(ns, int) else ns
    BM, BN, WM, WN, SA, SB, splits = r["bm"], r["bn"], r["wm"], r["wn"], r["sa"], r["sb"], r["splits"]
    NW = KERNEL_TILES[r["family"]]
    tail = not (k % 128 == 0 and k <= MAX_K and sum(ns) <= MAX_COLS)
    mat, local = own_tile(ns, BN)
    tm, tn = -(-m // BM), len(mat)
    T, G = tm * tn, tm * tn * splits
    assert r["grid_x"] == G and r["block"] == 64 * NW and (BM // WM) * (BN // WN) == NW
    assert len(ns) == 1 or (splits == 1 and not tail)
    assert not tail or (splits == 1 and NW == 4)
    KT = k // 128 + 1 if tail else k // 128 // splits
    assert tail or KT * splits * 128 == k
    LA, LB = BM // 8 // NW, BN // 8 // NW
    ASL, BSL = BM * 128, BN * 128
    assert SA * ASL + SB * BSL <= 160 * 1024
    Lt = xcd_slot(np.arange(G), G)
    split, Lt = Lt // T, Lt % T
    s0 = Lt // (STRIP * tn) * STRIP
    inside = Lt % (STRIP * tn)
    sm = np.minimum(STRIP, tm - s0)
    m0, tile = (s0 + inside % sm) * BM, inside // sm
    assert len({*zip(split.tolist(), m0.tolist(), tile.tolist())}) == G
    rotated = not tail and NW == 8 and splits == 1 and tn == 1 and T <= CUS
    for rot in {0, (T - 1) % KT if rotated else 0}:  # every chunk once, whatever the start
        assert np.array_equal(np.sort([kt + rot - (KT if kt + rot >= KT else 0) for kt in range(KT)]), np.arange(KT))
    kbase = split * KT * 128
    wave, lane = np.arange(NW)[:, None], np.arange(64)[None, :]
    chunk = lambda row: ((lane & 7) ^ ((row >> 1) & 7)) * 16  # noqa: E731
    slots = {"A": [], "B": []}
    for name, L, first, rows, pick in (("A", LA, m0, [m], np.zeros(G, int)), ("B", LB, local[tile] * BN, ns, mat[tile])):
        for j in range(L):
            row = 8 * (wave * L + j) + (lane >> 3)                               # [NW, 64]
            slots[name].append((wave * L + j) * 1024 + lane * 16)
            for i, size in enumerate(rows):
                f, kb = first[pick == i], kbase[pick == i]
                if f.size == 0:
                    continue
                assert f.max() < size  # the tile's first row exists: it stands in for rows past the end
                src = np.where(f[:, None, None] + row < size, row, 0) * k            # lane offset
                if not tail:
                    assert src.max() + chunk(row).max() < 1 << 32                    # held in 32 bits
                    at = f[:, None, None] * k + kb[:, None, None] + src + chunk(row)
                    within(f"gemm_dma {name}", at, at + (KT - 1) * 128 + 16, size * k)
                    continue
                for kt in (range(KT) if KT < 4 else (0, KT - 2, KT - 1)):
                    kk = kt * 128 + chunk(row)
                    at = f[:, None, None] * k + src + np.where(kk < k, kk, 0)  # activations past K: kZeroChunk
                    if name == "A":
                        at = at[:, kk < k]
                    within(f"gemm_dma {name} tail", at, at + 16, size * k)
    for name, size in (("A", ASL), ("B", BSL)):
        written_once(f"gemm_dma {name} ring slot", np.concatenate([s.ravel() for s in slots[name]]) // 16, size // 16)
    off = frag_offsets()
    wm0, wn0 = (np.arange(NW) // (BN // WN)) * WM, (np.arange(NW) % (BN // WN)) * WN
    for f in range(WM // 32):
        a = (wm0 + 32 * f)[:, None, None] * 128 + off[None]
        within("gemm_dma A fragments", a, a + 16, ASL)
    for f in range(WN // 32):
        b = (wn0 + 32 * f)[:, None, None] * 128 + off[None]
        within("gemm_dma B fragments", b, b + 16, BSL)
    for i, n in enumerate(ns):
        sel = np.flatnonzero(mat[tile] == i)
        n0 = local[tile[sel]] * BN
        assert tail or (4 * n + 31) * 4 < 1 << 32  # store_blocks' 32-bit lane offset
        rows, cols = store_blocks(m, n, m0[sel][:, None] + wm0[None, :], n0[:, None] + wn0[None, :], WM // 32, WN // 32)
        if splits == 1:
            written_once("gemm_dma out", rows * n + cols, m * n)
        else:
            # slab index of each store: repeat the per-workgroup split over its stores
            per_wg = [store_blocks(m, n, m0[w] + wm0, n0[w] + wn0, WM // 32, WN // 32) for w in range(G)]
            idx = np.concatenate([split[w] * m * n + rr * n + cc for w, (rr, cc) in enumerate(per_wg)])
            written_once("gemm_dma slabs", idx, splits * m * n)
            check_epilogue(m, n, r, residual)


def check_tall(m, ns, k, r, residual):
    """gemm_tall, one matrix or several: per-wave DMA instruction dealing, the
    rings, the two compute mappings, the stores."""
    ns = [ns] if isinstance(ns, int) else ns
    BN, SA, SB, MA, splits = r["bn"], r["sa"], r["sb"], r["ma"], r["splits"]
    FN, ASL, BSL, NB = BN // 32, MA * 128, BN * 128, BN // 8
    kMaxA, kMaxB = (MA // 8 + 7) // 8, (NB + 7) // 8
    assert SA * ASL + SB * BSL <= 160 * 1024 and m <= MA
    mat, local = own_tile(ns, BN)
    tn = len(mat)
    G = tn * splits
    assert r["grid_x"] == G and (len(ns) == 1 or splits == 1)
    KT = k // 128 // splits
    assert k % 128 == 0 and KT * splits * 128 == k
    Lt = xcd_slot(np.arange(G), G)
    split, pick, n0 = Lt // tn, mat[Lt % tn], local[Lt % tn] * BN
    width = np.asarray(ns)[pick]  # each workgroup's matrix: its columns
    kbase = split * KT * 128
    NA = -(-m // 8)
    for wave in range(8):
        na, nb = (NA + 7 - wave) // 8, (NB + 7 - wave) // 8
        assert na <= kMaxA and nb <= kMaxB
        lane = np.arange(64)
        for j in range(na):
            row = 8 * (wave + 8 * j) + (lane >> 3)
            assert row.max() < MA  # the ring slot row: 1024 (wave + 8 j) + 16 lane < MA * 128
            src = np.minimum(row, m - 1) * k + kbase[:, None] + ((lane & 7) ^ ((row >> 1) & 7)) * 16
            within("gemm_tall A", src, src + (KT - 1) * 128 + 16, m * k)
            dst = 1024 * (wave + 8 * j) + lane * 16
            within("gemm_tall A ring slot", dst, dst + 16, ASL)
        for j in range(nb):
            br = 8 * (wave + 8 * j) + (lane >> 3)
            src = (np.minimum(n0[:, None] + br, width[:, None] - 1) * k + kbase[:, None]
                   + ((lane & 7) ^ ((br >> 1) & 7)) * 16)
            assert src.min() >= 0 and (src + (KT - 1) * 128 + 16 <= (width * k)[:, None]).all(), "gemm_tall B"
            dst = 1024 * (wave + 8 * j) + lane * 16
            within("gemm_tall B ring slot", dst, dst + 16, BSL)
    off = frag_offsets()
    stores = []
    if MA == 64:
        T = -(-m // 32) * FN
        for wave in range(min(T, 8)):
            mb, nbk = wave // FN, wave % FN
            a = mb * 32 * 128 + off
            b = nbk * 32 * 128 + off
            within("gemm_tall A fragments", a, a + 16, ASL)
            within("gemm_tall B fragments", b, b + 16, BSL)
            stores.append((32 * mb + 0 * n0, n0 + 32 * nbk, 1, 1))
        assert T <= 8, "one 32 x 32 block per wave"
    else:
        for wave in range(8):
            if 32 * wave >= m:
                continue
            a = 32 * wave * 128 + off
            within("gemm_tall A fragments", a, a + 16, ASL)
            for jj in range(FN):
                b = 32 * jj * 128 + off
                within("gemm_tall B fragments", b, b + 16, BSL)
            stores.append((32 * wave + 0 * n0, n0, 1, FN))
    for i, n in enumerate(ns):
        idx = []
        for w in np.flatnonzero(pick == i):
            for (row0, col0, fm, fn) in stores:
                rr, cc = store_blocks(m, n, row0[w], col0[w], fm, fn)
                idx.append(split[w] * m * n + rr * n + cc)
        written_once("gemm_tall slabs" if splits > 1 else "gemm_tall out", np.concatenate(idx), splits * m * n)
    if splits > 1:
        check_epilogue(m, ns[0], r, residual)


def check_epilogue(m, n, r, residual):
    """splitk_epilogue / splitk_epilogue8 (gemm.hip): grid
    (ceil(n / cols / 256), min(m, 65535)), thread columns c .. c + cols - 1,
    rows blockIdx.y, + gridDim.y, ...; slab index clamped to splits - 1."""
    cols, splits = r["epi_cols"], r["splits"]
    assert n % cols == 0, "the epilogue works on whole column groups"
    gx, gy = -(-(n // cols) // 256), min(m, 65535)
    c = (np.arange(gx)[:, None] * 256 + np.arange(256)[None, :]).ravel() * cols
    c = c[c < n]
    rows = np.arange(m)  # row r is visited by blockIdx.y = r mod gy
    i = rows[:, None] * n + c[None, :]
    for s in range(4):  # kMaxSplits slab loads, clamped
        base = min(s, splits - 1) * m * n + i
        within("split-K epilogue slabs", base, base + cols, splits * m * n)
    within("split-K epilogue ws", c, c + cols, n)
    if residual:
        within("split-K epilogue residual", i, i + cols, m * n)
    written_once("split-K epilogue out", (i[..., None] + np.arange(cols)).ravel(), m * n)


def check_skinny(m, n, k, r):
    """gemm_skinny (gemm.hip): grid (ceil(n / 16), 1), S waves split K in
    64-byte steps; loads guarded by kk + koff < K (16-byte reads, K % 16 == 0)."""
    MT, S, U = r["mt"], r["s"], r["u"]
    assert r["grid_x"] == -(-n // 16) and r["grid_y"] == 1 and 16 * MT >= m and k % 16 == 0
    n0 = np.arange(r["grid_x"]) * 16
    steps = -(-k // 64)
    per = -(-steps // S)
    lane = np.arange(64)
    koff = (lane >> 4) * 16
    for wave in range(S):
        s0, s1 = min(wave * per, steps), min(wave * per + per, steps)
        for s in ({s0, s1 - 1} if s1 > s0 else set()):
            kk = s * 64
            ok = kk + koff < k
            wrow = np.minimum(n0[:, None] + (lane & 15), n - 1)
            src = (wrow * k + koff + kk)[:, ok]
            within("gemm_skinny W", src, src + 16, n * k)
            for t in range(MT):
                arow = t * 16 + (lane & 15)
                src = (arow * k + koff + kk)[ok & (arow < m)]
                within("gemm_skinny A", src, src + 16, m * k)
    # epilogue: thread i -> (t, v, l); r = m0 + 16 t + 4 (l >> 4) + v, c = n0 + (l & 15)
    i = np.arange(MT * 4 * 64)
    l, v, t = i & 63, (i >> 6) & 3, i >> 8
    rr = t * 16 + 4 * (l >> 4) + v
    cc = n0[:, None] + (l & 15)
    rr = np.broadcast_to(rr, cc.shape)
    keep = (rr < m) & (cc < n)
    written_once("gemm_skinny out", rr[keep] * n + cc[keep], m * n)


def check_narrow(m, ns, k, r):
    """gemm_narrow, one matrix or several: ceil(n / (16 NB)) workgroups of 64 S
    threads per matrix (NB = 2 for groups only); wave w sums ST = K / (128 S) of
    the 128-byte K chunks through its own R-stage ring: at S = 4 stage s reads
    chunk w ST + s, at S = 8 chunk ((s + b) mod ST) S + w for workgroup b; the
    chunks of all waves and stages of a workgroup must be every chunk of K
    exactly once.  DMA instruction j < 2 NB + LAL fills rows 8j .. 8j + 7 of a
    stage (lane l: row 8j + l / 8, 16-byte piece (l % 8) ^ (row % 8)); rows below
    16 NB are weight rows n0 + row clamped to n - 1, the others activation rows
    row - 16 NB, loaded only below M."""
    single = isinstance(ns, int)
    ns = [ns] if single else ns
    MB, S, LAL, R = r["mt"], r["s"], r["u"], r["sa"]
    NB = 1 if single else r["bn"] // 16
    mat, local = own_tile(ns, 16 * NB)
    assert r["grid_x"] == len(mat) and r["grid_y"] == 1 and r["block"] == 64 * S and r["splits"] == 1
    assert k % (128 * S) == 0 and 16 * MB >= m
    # every row below M has its DMA instruction, and every issued instruction has a live lane
    assert 8 * LAL >= m and 8 * (LAL - 1) < m, (m, LAL)
    ROWS, L = 16 * (NB + MB), 2 * NB + LAL
    STAGE, RING = ROWS * 128, R * ROWS * 128
    assert L <= ROWS // 8 and S * RING <= 160 * 1024 and (R - 1) * L < 64
    ST = k // (128 * S)
    n0 = (local * 16 * NB)[:, None]
    width = np.asarray(ns)[mat][:, None]
    lane = np.arange(64)
    b = np.arange(r["grid_x"])

    def kchunk(wave, st):
        """K chunk of stage st of wave `wave`, per workgroup."""
        if S >= 8:
            return ((st + b) % ST) * S + wave
        return np.full(b.shape, wave * ST + st)

    seen = np.zeros((r["grid_x"], k // 128), np.int64)
    for wave in range(S):
        for st in range(ST):
            np.add.at(seen, (b, kchunk(wave, st)), 1)
    assert (seen == 1).all(), "every K chunk exactly once per workgroup"
    for wave in range(S):
        for st in ({0, ST - 1} if ST > 0 else set()):
            for j in range(L):
                row = 8 * j + (lane >> 3)
                chunk = ((lane & 7) ^ (row & 7)) * 16
                koff = kchunk(wave, st)[:, None] * 128 + chunk
                if j < 2 * NB:
                    src = np.minimum(n0 + row, width - 1) * k + koff
                    assert src.min() >= 0 and (src + 16 <= width * k).all(), "gemm_narrow W"
                else:
                    g = row - 16 * NB
                    live = g < m
                    src = (g * k + koff)[:, live]
                    within("gemm_narrow A", src, src + 16, m * k)
                dst = wave * RING + (st % R) * STAGE + j * 1024 + lane * 16
                within("gemm_narrow LDS DMA", dst, dst + 16, S * RING)
    fr, fq = lane & 15, lane >> 4
    for h in range(2):
        c = 4 * h + fq
        for block in range(NB + MB):  # NB weight blocks, then MB activation blocks
            row = 16 * block + fr
            a = row * 128 + ((c ^ (row & 7)) * 16)
            within("gemm_narrow fragments", a, a + 16, STAGE)
    # reduction slot of value v of block (t, u) of a wave, and its reader: index i of every wave
    t, u, v = np.meshgrid(np.arange(MB), np.arange(NB), np.arange(4), indexing="ij")
    red = (((np.arange(S)[:, None, None, None, None] * MB + t[..., None]) * NB + u[..., None]) * 4 + v[..., None]) * 64 \
        + lane
    written_once("gemm_narrow reduction", red, S * MB * NB * 256)
    within("gemm_narrow reduction", red * 4, red * 4 + 4, S * RING)
    i = np.arange(MB * NB * 4 * 64)
    l, v, u, t = i & 63, (i >> 6) & 3, (i >> 8) % NB, (i >> 8) // NB
    assert np.array_equal(((t * NB + u) * 4 + v) * 64 + l, i)
    for x, n in enumerate(ns):
        rr = 16 * t + 4 * (l >> 4) + v
        cc = n0[mat == x] + 16 * u + (l & 15)
        rr = np.broadcast_to(rr, cc.shape)
        keep = (rr < m) & (cc < n)
        written_once("gemm_narrow out", rr[keep] * n + cc[keep], m * n)


# ------------------------------------------------------------------ GEMV routes
def check_gemv_m1(m, n, k, r, residual, argmax=False):
    """gemv_m1_one / gemv_m1 (gemv.hip): wave g owns rows R g ..
    R g + R - 1; loads clamped to n - 1; lanes < R store rows < n."""
    R, KC, W = r["rows"], r["kc"], r["waves"]
    assert m == 1 and k == KC * 1024
    groups = -(-n // R)
    assert r["grid_x"] == -(-groups // W)
    g = np.arange(r["grid_x"] * W)
    live = g < groups
    row0 = np.where(live, g * R, 0)
    lane = np.arange(64)
    within("gemv q", lane * 16, lane * 16 + 16 + (KC - 1) * 1024, k)
    erow = np.minimum(row0[:, None] + np.minimum(lane, R - 1), n - 1)
    within("gemv ws / residual", erow, erow + 1, n)
    for rr in range(R):
        src = np.minimum(row0 + rr, n - 1)[:, None] * k + lane * 16
        within("gemv W", src, src + (KC - 1) * 1024 + 16, n * k)
    row = row0[:, None] + lane
    keep = live[:, None] & (lane < R) & (row < n)
    written_once("gemv out", row[keep], n)
    if argmax:
        # one key per workgroup into a workspace of argmax_keys_for(n) keys
        assert r["grid_x"] <= -(-n // 4), "selection keys exceed the workspace bound"


def check_gemv_mt(m, n, k, r, residual):
    """gemv_mt (gemv.hip): 4-row groups, MT activation rows per pass
    (blockIdx.y), 1 KiB chunks with rotation, loads guarded by kk < K."""
    MT, R = r["mt"], 4
    groups = -(-n // R)
    assert r["grid_x"] == -(-groups // 4) and r["grid_y"] == -(-m // MT)
    g = np.arange(r["grid_x"] * 4)
    live = g < groups
    row0 = np.where(live, g * R, 0)
    lane = np.arange(64)
    nch = -(-k // 1024)
    for ci in {0, nch - 1}:
        kk = ci * 1024 + lane * 16
        ok = kk < k
        for rr in range(R):
            src = (np.minimum(row0 + rr, n - 1)[:, None] * k + kk)[:, ok]
            within("gemv_mt W", src, src + 16, n * k)
        m0 = np.arange(r["grid_y"]) * MT
        for t in range(MT):
            xr = m0 + t
            src = (np.where(xr < m, xr, 0)[:, None] * k + kk)[xr < m][:, ok]
            within("gemv_mt q", src, src + 16, m * k)
    V = R * MT
    m0 = np.arange(r["grid_y"]) * MT
    t = m0[:, None, None] + (lane // R)[None, None, :]
    row = row0[None, :, None] + (lane % R)[None, None, :]
    t, row = np.broadcast_arrays(t, row)
    keep = live[None, :, None] & (lane < V)[None, None, :] & (row < n) & (t < m)
    written_once("gemv_mt out", (t * n + row)[keep], m * n)


def check_linear(m, n, k, dtype=BF16, residual=False, path=AUTO, workspace=0):
    r = route(m, n, k, dtype, residual, path, workspace)
    fam = r["family"]
    if fam in (1, 2):
        check_gemv_m1(m, n, k, r, residual)
    elif fam == 3:
        check_gemv_mt(m, n, k, r, residual)
    elif fam == 11:
        check_skinny(m, n, k, r)
    elif fam == 12:
        check_tall(m, n, k, r, residual)
    elif fam in KERNEL_TILES:
        check_dma(m, n, k, r, residual)
    elif fam == 15:
        check_narrow(m, n, k, r)
    else:
        raise AssertionError(f"no route for {(m, n, k)}: {r}")
    return r


def grouped_route(m, ns, k):
    r, n = np.zeros(ROUTE_LEN, np.int32), np.asarray(ns, np.uint64)
    assert _lib.lib().w8a8_diag_grouped_route(m, k, len(ns), n.ctypes.data, r.ctypes.data, ROUTE_LEN) == 0
    keys = ("family grid_x grid_y block bm bn wm wn sa sb ma mt s u splits nt epi_cols rows kc waves").split()
    return dict(zip(keys, (int(v) for v in r)))


def check_grouped(m, ns, k):
    """The one launch over the matrices that have columns, or each matrix's own."""
    r, ns = grouped_route(m, ns, k), [n for n in ns if n]
    if r["family"] == 15:
        check_narrow(m, ns, k, r)
    elif r["family"] == 12:
        check_tall(m, ns, k, r, False)
    elif r["family"] in KERNEL_TILES:
        check_dma(m, ns, k, r, False)
    elif r["family"] == 0:
        assert m > 4
        for n in ns:
            check_linear(m, n, k, path=MFMA)
    else:
        assert r["family"] in (2, 3) and m <= 4  # the dot4 launch: each matrix's row groups, as for one
    return r


# ------------------------------------------------------------------ tests
@pytest.mark.parametrize("n,k", DECODE)
def test_decode_shapes_m1(n, k):
    """C1 / C2: the decode projections at M = 1, and with a residual."""
    for residual in (False, True):
        r = check_linear(1, n, k, residual=residual)
        assert r["family"] == 1


def test_lm_head_argmax():
    """C3: the 151,936-row head's fused-selection GEMV."""
    n, k = 151936, 4096
    r = argmax_route(n, k)
    assert r["family"] == 2 and r["waves"] == 16
    check_gemv_m1(1, n, k, r, False, argmax=True)
    for nn in (1, 3, 4097, 50000):
        check_gemv_m1(1, nn, k, argmax_route(nn, k), False, argmax=True)


@pytest.mark.parametrize("m", [129, 512])
@pytest.mark.parametrize("n,k", DECODE)
def test_prefill_shapes(m, n, k):
    """C4: M = 129 and 512 on the four layer shapes, with and without the
    split-K workspace, plain and with a residual."""
    for path in (AUTO, MFMA):
        for ws in (0, workspace_bytes(m, n, k)):
            for residual in (False, True):
                check_linear(m, n, k, residual=residual, path=path, workspace=ws)


@pytest.mark.parametrize("m", [130, 131, 135, 136, 140, 159])
@pytest.mark.parametrize("n,k", DECODE)
def test_m129_tails(m, n, k):
    """The rows past a 32-row block and past the 128-row tile: M = 129-135
    and 136-159 (sampled)."""
    check_linear(m, n, k, path=MFMA, workspace=workspace_bytes(m, n, k))
    check_linear(m, n, k, residual=True)


@pytest.mark.parametrize("m", [4, 16, 64])
@pytest.mark.parametrize("n,k", [(24576, 4096), (4096, 12288)])
def test_ragged_small_m(m, n, k):
    """C5: the ragged batches on gate_up and down, on both families."""
    for path in (DOT4, MFMA):
        for ws in (0, workspace_bytes(m, n, k)):
            check_linear(m, n, k, path=path, workspace=ws)


@pytest.mark.parametrize("m", [2, 3, 7, 8, 17, 33, 65, 100, 200, 255, 256, 257, 300])
def test_other_m_and_n_not_multiple_of_96(m):
    """Every family at M between the configurations, with N % 96 != 0 (and
    not a multiple of 64 or 16 where the routes allow it)."""
    for n, k in [(4000, 4096), (6100, 4096), (24500, 4096), (1000, 12288), (4100, 4096)]:
        for ws in (0, workspace_bytes(m, n, k)):
            check_linear(m, n, k, workspace=ws)
        check_linear(m, n, k, path=MFMA, workspace=workspace_bytes(m, n, k))
        check_linear(m, n, k, residual=True)


@pytest.mark.parametrize("m,n,k", [(100, 4096, 4112), (300, 1000, 1040), (65, 777, 2064), (1, 5000, 1040),
                                   (3, 333, 48)])
def test_k_not_multiple_of_128(m, n, k):
    """gemm_dma with a K tail, gemm_skinny and gemv_mt at odd K."""
    check_linear(m, n, k)
    check_linear(m, n, k, path=DOT4)


@pytest.mark.parametrize("n,k", [(4096, 4096), (6144, 4096), (4096, 12288), (1000, 512), (4100, 8192), (333, 2048),
                                 (17, 12288)])
def test_narrow_every_m(n, k):
    """gemm_narrow at every M it takes (1-16, and 17-64 at K <= 4096 on
    N <= 4096): both wave counts (K below and from 8192), one to eight live
    activation loads per stage, N not a multiple of 16, a one-stage slice
    (K = 512)."""
    took = 0
    for m in [*range(1, 34), 40, 41, 47, 48, 49, 56, 57, 63, 64]:
        for path in (AUTO, MFMA):
            r = check_linear(m, n, k, path=path, workspace=workspace_bytes(m, n, k))
            if path == MFMA and m <= 16:
                assert r["family"] == 15, (m, n, k, r)
            took += r["family"] == 15
    assert took >= 16


@pytest.mark.parametrize("m,n,k", seeded_linear_shapes())
def test_seeded_shape_sweep(m, n, k):
    """The shapes of the GPU sweep (test_gpu_parity.test_linear_seeded_shape_sweep),
    replayed first here on every path it runs: AUTO with and without the
    split-K workspace, BF16 and f32 with the residual; the dot4 GEMV and
    the MFMA family forced."""
    wsb = workspace_bytes(m, n, k)
    for path in (AUTO, DOT4, MFMA):
        for workspace in ((0, wsb) if path != DOT4 else (0,)):
            check_linear(m, n, k, path=path, workspace=workspace)
            check_linear(m, n, k, F32, residual=True, path=path, workspace=workspace)
    check_linear(m, n, k, I32, path=MFMA, workspace=wsb)


@pytest.mark.parametrize("m,n,k,skinny", [
    (17, 1024, 8192, True), (32, 512, 16000, True), (32, 4096, 8192, True), (32, 4100, 8192, False),
    (33, 1024, 8192, False), (64, 1024, 12304, True), (64, 4096, 2064, True), (64, 4100, 2064, False),
    (65, 1024, 12304, False), (24, 8192, 1040, True), (25, 8192, 1040, False), (32, 8192, 528, True),
    (24, 8208, 528, False), (33, 8192, 528, False), (48, 8192, 384, True), (49, 8192, 384, False),
    (48, 4096, 896, True), (48, 4096, 1152, False), (64, 4096, 384, True), (64, 4096, 640, False)])
def test_k_split_over_waves_on_narrow_n(m, n, k, skinny):
    """Where no plan runs (K tails, no workspace): gemm_skinny up to one
    workgroup per CU, gemm_dma's small tiles beyond."""
    assert (check_linear(m, n, k, path=MFMA)["family"] == 11) == skinny


@pytest.mark.parametrize("m,n,k", [(129, 8192, 4096), (256, 4096, 4096), (193, 6144, 2048), (33000, 64, 8192)])
def test_auto_ignores_a_workspace_that_only_slows_it(m, n, k):
    """The launch follows the shape, not the pointer: with a workspace for the
    split plan AUTO runs the same route as without one, and MFMA splits."""
    ws = workspace_bytes(m, n, k)
    assert ws > 0
    assert route(m, n, k, workspace=ws) == route(m, n, k) and route(m, n, k)["splits"] == 1
    assert route(m, n, k, path=MFMA, workspace=ws)["splits"] > 1


@pytest.mark.parametrize("m,n,k,split", [(64, 4096, 4096, True), (49, 4096, 4096, True), (48, 4096, 4096, False),
                                         (53, 3584, 4096, True), (52, 3584, 4096, False),
                                         (53, 1024, 4096, True), (52, 1024, 4096, False),
                                         (57, 1536, 4096, True), (56, 1536, 4096, False), (64, 4096, 3584, False),
                                         (64, 2560, 4096, False),
                                         (64, 4095, 4096, False), (40, 4096, 4096, False)])
def test_split_k_past_the_narrow_kernel(m, n, k, split):
    """At the most rows and the longest K of gemm_narrow a workspace gives
    split K, which is faster there; without one the shape stays narrow."""
    assert (workspace_bytes(m, n, k) > 0) == split
    r = check_linear(m, n, k, workspace=workspace_bytes(m, n, k))
    assert r["family"] == (12 if split else 15) and r["splits"] == (4 if split else 1)
    assert check_linear(m, n, k)["family"] == 15


GROUPS = [(200, 33, 1), (64, 0, 96, 31), (4096, 1024, 1024), (4100, 33, 1, 7), (12288, 12288), (10000, 11600, 5)]


@pytest.mark.parametrize("m", [2, 4, 5, 16, 17, 32, 33, 48, 64, 65, 129, 160, 161, 256, 257, 512])
@pytest.mark.parametrize("ns", GROUPS)
def test_grouped_launches(m, ns):
    """Sibling projections: one GEMM launch over the matrices' column tiles,
    each tile inside its own matrix; every route and both gemm_narrow widths."""
    for k in (512, 1024, 4096, 8192):
        check_grouped(m, ns, k)


def test_every_grouped_route_is_replayed():
    """gemm_narrow on 16 and 32 columns, the one-M-tile kernel, gemm_dma with
    eight and four waves, the dot4 launch, and one launch per matrix."""
    seen = {(r["family"], r["bn"] if r["family"] == 15 else 0)
            for r in (check_grouped(m, ns, k) for m, ns, k in [
                (16, (200, 33), 512), (64, (4096, 1024, 1024), 4096), (129, (12288, 12288), 4096),
                (512, (4096, 1024, 1024), 4096), (100, (300, 40), 4096), (2, (300, 40), 1040), (70, (100, 33), 1040)])}
    assert seen == {(15, 16), (15, 32), (12, 0), (13, 0), (14, 0), (3, 0), (0, 0)}, seen


@pytest.mark.parametrize("m,ns,k,gemm", [
    (2, (4096, 1024, 1024), 4096, True), (2, (8192, 2048, 2048), 4096, False), (2, (8192, 8192), 1024, False),
    (2, (2048, 1024, 1024), 2048, True), (2, (4096, 2048, 2048), 3072, False), (2, (12288, 12288), 4096, True),
    (2, (2048, 512, 512), 12288, True), (2, (4096, 1024, 1024), 8192, False), (2, (1024, 512, 512), 16384, False),
    (3, (2048, 1024, 1024), 12288, True), (3, (8192, 8192), 8192, False), (3, (8192, 2048, 2048), 2048, False),
    (3, (4096, 4096), 2048, True), (4, (4096, 1024, 1024), 9216, True), (4, (4096, 4096), 16384, False),
    (4, (8192, 8192), 4096, True), (4, (8192, 8192), 2048, False), (4, (100, 33), 1040, False)])
def test_grouped_gemm_or_dot4(m, ns, k, gemm):
    """Two to four rows of siblings: the launch that was faster with distinct
    weights, gemm_narrow (or the 96-column tiles) or one dot4 GEMV."""
    assert (check_grouped(m, ns, k)["family"] >= 11) == gemm


@pytest.mark.parametrize("tile,family,m,n,k", [((64, 64), 14, 150, 515, 1280), ((64, 64), 14, 65, 33, 16),
                                               ((64, 64), 14, 257, 515, 1392), ((128, 64), 14, 1025, 2003, 16),
                                               ((128, 128), 14, 1300, 3003, 144), ((256, 128), 14, 2049, 2003, 1296),
                                               ((256, 256), 13, 2049, 6003, 1280), ((64, 128), 13, 129, 10003, 1280),
                                               ((128, 64), 13, 22000, 60, 640), ((256, 256), 14, 1300, 6003, 1296)])
def test_every_dma_tile(tile, family, m, n, k):
    """gemm_dma's tiles, several strips of M tiles, ragged edges, K tails of
    16 bytes and more, one column of tiles (rotated K)."""
    r = check_linear(m, n, k)
    assert (r["family"], r["bm"], r["bn"]) == (family, *tile)


def test_every_family_is_replayed():
    """The shapes above reach every GEMM and GEMV family."""
    seen = set()
    for (m, n, k, ws) in [(1, 4096, 4096, 0), (1, 4096, 1040, 0), (3, 4096, 4096, 0), (3, 4096, 1040, 0),
                          (129, 4096, 12288, 1 << 30), (512, 24576, 4096, 0), (100, 4096, 4112, 0)]:
        seen.add(route(m, n, k, workspace=ws)["family"])
    seen.add(argmax_route(4096, 4096)["family"])
    assert seen == {1, 2, 3, 11, 12, 13, 14, 15}, seen


# ------------------------------------------------------------------ folded producers
def check_rows_split(n, NS, RS, K):
    """gemv_m1_split / gemv_rowtail_split streaming waves (gemv.hip): row r of
    wave wv of workgroup b is (r NS + wv) G + slot(b),
    loads clamped to n - 1, stores guarded by row < n."""
    G = -(-n // (NS * RS))
    b, wv, rr = np.meshgrid(np.arange(G), np.arange(NS), np.arange(RS), indexing="ij")
    row = (rr * NS + wv) * G + xcd_slot(b, G)
    er = np.minimum(row, n - 1)
    lane = np.arange(64)
    src = er[..., None] * K + lane * 16
    within("split W", src, src + K - 1024 + 16, n * K)
    written_once("split out", row[row < n], n)


def check_swiglu_split(n, NS=12, CS=4):
    """gemv_swiglu_split (gemv.hip): coordinate k of wave wv of
    workgroup b is (k NS + wv) G + slot(b)."""
    G = -(-n // (NS * CS))
    b, wv, kk = np.meshgrid(np.arange(G), np.arange(NS), np.arange(CS), indexing="ij")
    c = (kk * NS + wv) * G + xcd_slot(b, G)
    src = np.minimum(c, n - 1)[..., None] * 4096 + np.arange(64) * 16
    within("swiglu split W", src, src + 3 * 1024 + 16, n * 4096)
    written_once("swiglu split out", c[c < n], n)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 1000, 4095, 4096, 4097, 5000, 6143, 6144, 6145, 24576, 40000])
def test_folded_producer_rows(n):
    """Every row of the folded-producer GEMVs written once, every weight load
    inside the matrix: 8 streaming waves x 2 rows up to N = 4096 and 12 x 2
    beyond (K = 4096), 8 x 2 for the down fold (K = 12,288)."""
    check_rows_split(n, 8 if n <= 4096 else 12, 2, 4096)
    check_rows_split(n, 8, 2, 12288)


@pytest.mark.parametrize("n", [1, 47, 48, 49, 4096, 12287, 12288, 12289, 30000])
def test_swiglu_split_coordinates(n):
    check_swiglu_split(n)


def test_producer_row_layout():
    """The producer waves' row loads: thread pt of the four reads x[pt + 256 i]
    (i < 16) of a 4096-wide row, and for the down fold elements
    4 (pt + 256 j) .. + 3 (j < 12) of the 12,288-wide act row; codes go to
    LDS byte pt + 256 i, or word pt + 256 j."""
    pt = np.arange(256)[:, None]
    x = pt + 256 * np.arange(16)
    written_once("producer row", x, 4096)
    e = 4 * (pt + 256 * np.arange(12))
    written_once("rowtail act", (e[..., None] + np.arange(4)).ravel(), 12288)


# ------------------------------------------------------------------ planted mistakes
def test_checker_catches_planted_mistakes():
    """The checks above must fail on the mistakes they exist for: a tail row
    read without its clamp, a store written twice or not at all, a slot
    mapping off by one."""
    m, n, k = 129, 4096, 4096
    r = route(m, n, k, path=MFMA, workspace=workspace_bytes(m, n, k))
    assert r["family"] == 12  # gemm_tall, 160-row tile, split K
    lane = np.arange(64)
    row = 8 * (0 + 8 * 2) + (lane >> 3)  # wave 0's third activation row group: rows 128-135
    KT = k // 128 // r["splits"]
    unclamped = row * k + ((lane & 7) ^ ((row >> 1) & 7)) * 16 + (r["splits"] - 1) * KT * 128
    with pytest.raises(AssertionError, match="past the buffer"):
        within("unclamped A", unclamped, unclamped + (KT - 1) * 128 + 16, m * k)
    clamped = np.minimum(row, m - 1) * k + ((lane & 7) ^ ((row >> 1) & 7)) * 16 + (r["splits"] - 1) * KT * 128
    within("clamped A", clamped, clamped + (KT - 1) * 128 + 16, m * k)
    with pytest.raises(AssertionError):
        written_once("duplicate", np.array([0, 1, 1, 3]), 4)
    with pytest.raises(AssertionError):
        written_once("missing", np.array([0, 1, 3]), 4)
    # folded-producer rows with the slot shifted by one workgroup
    n, NS, RS = 6144, 12, 2
    G = -(-n // (NS * RS))
    b, wv, rr = np.meshgrid(np.arange(G), np.arange(NS), np.arange(RS), indexing="ij")
    bad = (rr * NS + wv) * G + (xcd_slot(b, G) + 1)
    with pytest.raises(AssertionError):
        written_once("shifted rows", bad[bad < n], n)
    # a 32 x 32 MFMA block's value layout with the half-wave term dropped
    lane2 = np.arange(64)[:, None]
    v = np.arange(16)[None, :]
    wrong = (v >> 2) * 8 + (v & 3) + 0 * lane2
    with pytest.raises(AssertionError):
        written_once("block rows", (wrong * 32 + (lane2 & 31)).ravel(), 32 * 32)
    rows, cols = mfma32_rows_cols(lane2, v)
    written_once("block rows", (rows * 32 + np.broadcast_to(cols, rows.shape)).ravel(), 32 * 32)
    # gemm_narrow: activation rows loaded without the live mask (M = 3: rows 3-7 of the first
    # activation instruction), and a live-load count one short of the rows (M = 9, LAL = 1)
    m, n, k = 3, 4096, 4096
    r = route(m, n, k, path=MFMA)
    assert r["family"] == 15
    g = (8 * 2 + (lane >> 3)) - 16
    src = g * k + ((lane & 7) ^ ((g + 16) & 7)) * 16 + (r["s"] - 1) * (k // r["s"])
    with pytest.raises(AssertionError, match="past the buffer"):
        within("unmasked A", src, src + (k // r["s"] - 128) + 16, m * k)
    bad = dict(route(9, n, k, path=MFMA), u=1)
    with pytest.raises(AssertionError):
        check_narrow(9, n, k, bad)
    # gemm_dma: a four-wave tile dealt as if to eight waves, a tile count of another tile, and a
    # tail read that takes the weights' chunk past K
    r = route(150, 515, 1280)
    with pytest.raises(AssertionError):
        check_dma(150, 515, 1280, dict(r, family=13, block=512), False)
    with pytest.raises(AssertionError):
        check_dma(150, 515, 1280, dict(r, bn=128), False)
    k = 1040
    past = (514 * k) + 8 * 128 + ((lane & 7) ^ 0) * 16  # stage 8 of the last row, unclamped
    with pytest.raises(AssertionError, match="past the buffer"):
        within("unclamped tail", past, past + 16, 515 * k)
    # grouped: a tile given to the next matrix
    mat, local = own_tile([200, 33], 64)
    assert mat.tolist() == [0, 0, 0, 0, 1] and local.tolist() == [0, 1, 2, 3, 0]
    with pytest.raises(AssertionError):
        check_narrow(2, [200, 33], 512, dict(grouped_route(2, [200, 33], 512), bn=32))
