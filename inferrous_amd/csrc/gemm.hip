// gemm.hip -- INT8 MFMA GEMM (exact i32 accumulate) for prefill and small
// batches, with the fused per-token x per-channel dequant epilogue.
//
// Reference semantics (crates/inferrous-qwen3/): the M > 1 projections
//   linear_prefill src/kernels.rs:846-931, linear_splitk :932-1034,
//   linear_tiled :1035-1141, linear_large :1142-1289, epilogues
//   :918-930, :1008-1033, :1123-1140, :1249-1288:
//   out[r][c] = bf(RN(RN(f32(sum_k q[r][k] w[c][k]) * asc[r]) * ws[c]))
//
// gfx950 design.  Any k permutation applied identically to A and B leaves
// the exact integer sum unchanged, so each kernel reads both operands with
// one lane -> k map of its own choosing.  Layouts of the two matrix-core
// ops used:
//   v_mfma_i32_16x16x64_i8: per lane a 16-byte A fragment (row lane%16) and
//     a 16-byte B fragment (column lane%16); the 4 x i32 result of lane l
//     holds rows 4*(l/16)+v, column l%16.
//   v_mfma_i32_32x32x32_i8: 16-byte fragments, row / column lane%32; the
//     16 x i32 result of lane l holds rows 8*(v/4)+4*(l/32)+v%4, column l%32.
//
// Kernels:
//  * gemm_dma: the prefill GEMM, and every shape above 16 rows that no kernel
//    below takes; built on v_mfma_i32_32x32x32_i8 (on gfx950 the 16x16x64 int8
//    form issues at half its rate), eight waves per workgroup (two per SIMD,
//    so one wave's LDS reads overlap the other's MFMAs; four on the 64 x 64
//    tile and for k % 128 != 0).  Operands move global -> LDS with
//    global_load_lds_dwordx4 (no VGPR staging) in 128-byte K stages (whole
//    cache lines) through two rings, activations and weights, the weights
//    requested further ahead, the requests spread between the MFMAs; one
//    barrier per stage; the 16-byte chunks of each LDS row are XOR-swizzled so
//    fragment reads spread over the banks.  Workgroups are numbered XCD-aware
//    (below).  Tile shape per problem by measured cost.  With a caller
//    workspace, some shapes run split-K (i32 slabs + splitk_epilogue).
//  * gemm_tall (M <= 256, k % 128 == 0, where its plan applies; M tiles of
//    64, 160 or 256 rows): one M tile holds every activation row, so each
//    weight tile streams from HBM once; the waves hold 32 x 32 output blocks
//    one each (M <= 64) or 32-row slices of all BN columns, and those
//    holding none only move data; activation rows past M are never loaded;
//    split-K on narrow n.
//  * gemm_narrow (M <= 16, or M <= 64 on n <= 4096 at k <= 4096, where the
//    n / 96 tiles are fewer than 224 and k splits into S slices of 128-byte
//    stages): one workgroup owns 16 weight rows; its S waves split K
//    (contiguous slices at S = 4, interleaved 128-byte chunks at S = 8), and
//    each wave streams its share through its own global -> LDS ring (16 weight rows and the live activation rows of a 128-byte stage,
//    global_load_lds_dwordx4: eight whole lines per instruction), so the K
//    loop has no workgroup barrier and no split-K slabs leave the CU.  The S
//    partial 16 x 16 tiles are summed through LDS (exact) and stored by the
//    fused epilogue.
//  * gemm_skinny (M <= 16, and up to 64 on narrow n, where gemm_narrow and
//    gemm_tall do not run: k not in their stages, or a split-K plan without a
//    workspace; HBM-bound, 16x16x64 MFMA): one workgroup owns 16 weight rows; its S waves split K and stream
//    their weight fragments straight from HBM into MFMA B operands (no LDS
//    round trip), activation fragments come from L1/L2.  Partial i32 tiles
//    are summed through LDS -- exact.
#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "internal.hpp"

namespace w8a8 {

__device__ __forceinline__ v4i mfma16(v4i a, v4i b, v4i c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ void epilogue_store(const GemmArgs& a, uint32_t r, uint32_t c, int32_t acc) {
  const size_t o = (size_t)r * a.n + c;
  if (a.out_dtype == W8A8_OUT_I32) {
    reinterpret_cast<int32_t*>(a.out)[o] = acc;
    return;
  }
  const float v = dequant(acc, a.asc[r], a.ws[c]);
  if (a.out_dtype == W8A8_OUT_F32) {
    if (a.out) reinterpret_cast<float*>(a.out)[o] = v;
    if (a.residual) reinterpret_cast<float*>(a.combined)[o] = bf16_rne(a.residual[o] + v);
  } else {
    if (a.out) reinterpret_cast<uint16_t*>(a.out)[o] = (uint16_t)(__float_as_uint(v) >> 16);
    if (a.residual)
      reinterpret_cast<uint16_t*>(a.combined)[o] =
          (uint16_t)(__float_as_uint(bf16_rne(a.residual[o] + v)) >> 16);
  }
}

// ---------------------------------------------------------------- skinny
template <int MT, int S, int U>
__global__ __launch_bounds__(64 * S) void gemm_skinny(GemmArgs a) {
  __shared__ int red[S][MT][4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t n0 = blockIdx.x * 16;
  const uint32_t m0 = blockIdx.y * 16 * MT;
  const uint32_t K = a.k;
  const uint32_t steps = (K + 63) / 64;
  const uint32_t per = (steps + S - 1) / S;
  const uint32_t s0 = min(wave * per, steps), s1 = min(s0 + per, steps);
  const uint32_t koff = (lane >> 4) * 16;
  const int8_t* wp = a.w + (size_t)min(n0 + (lane & 15), a.n - 1) * K + koff;
  const int8_t* ap[MT];
  bool aok[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const uint32_t r = m0 + t * 16 + (lane & 15);
    aok[t] = r < a.m;
    ap[t] = a.q + (size_t)(aok[t] ? r : 0) * K + koff;
  }
  v4i acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = v4i{0, 0, 0, 0};
  for (uint32_t s = s0; s < s1; s += U) {
    v4i wv[U], av[U][MT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t kk = (s + u) * 64;
      const bool ok = (s + u < s1) && (kk + koff < K);
      wv[u] = ok ? load_nt16(wp + kk) : v4i{0, 0, 0, 0};
#pragma unroll
      for (int t = 0; t < MT; ++t) av[u][t] = (ok && aok[t]) ? load16(ap[t] + kk) : v4i{0, 0, 0, 0};
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t] = mfma16(av[u][t], wv[u], acc[t]);
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][t][v][lane] = acc[t][v];
  __syncthreads();
  for (int i = threadIdx.x; i < MT * 4 * 64; i += 64 * S) {
    const int l = i & 63, v = (i >> 6) & 3, t = i >> 8;
    int sum = 0;
#pragma unroll
    for (int w = 0; w < S; ++w) sum += red[w][t][v][l];
    const uint32_t r = m0 + t * 16 + 4 * (l >> 4) + v;
    const uint32_t c = n0 + (l & 15);
    if (r < a.m && c < a.n) epilogue_store(a, r, c, sum);
  }
}

// ---------------------------------------------------------------- dma
typedef int v16i __attribute__((ext_vector_type(16)));

__device__ __forceinline__ v16i mfma32(v4i a, v4i b, v16i c) {
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// s_waitcnt with vmcnt = N and the other counters left at their maximum
// (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] << 14).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}


#define W8A8_LDS_PTR(p) ((void __attribute__((address_space(3)))*)(p))

// Epilogue modes, resolved at compile time so the unrolled store loop stays
// branch-free: raw accumulators, f32 or BF16 outputs, each optionally with
// the residual sum bf(residual + out).  EP_SLAB is EP_I32 for a split-K slab
// that is streamed: non-temporal stores, read back once by the slab epilogue.
enum { EP_I32 = 0, EP_F32 = 1, EP_BF16 = 2, EP_F32_RES = 3, EP_BF16_RES = 4, EP_SLAB = 5 };
constexpr bool raw_i32(int ep) { return ep == EP_I32 || ep == EP_SLAB; }

// Grouped launches (GROUP): the matrix that owns column tile t becomes the
// launch's only one (a.w, a.ws, a.out, a.n), and the tile's index within it is
// returned.  Every boundary and operand sits at a fixed kernel-argument
// offset, so this is a batch of scalar loads, compares and selects.
struct NoGroup {};
template <bool GROUP>
using GroupArg = std::conditional_t<GROUP, GemmGroup, NoGroup>;

__device__ __forceinline__ uint32_t own_tile(GemmArgs&, const NoGroup&, uint32_t t) { return t; }
__device__ __forceinline__ uint32_t own_tile(GemmArgs& a, const GemmGroup& g, uint32_t t) {
  a.w = g.w[0], a.ws = g.ws[0], a.out = g.out[0], a.n = g.n[0];
  uint32_t first = 0;
#pragma unroll
  for (int i = 1; i < kMaxGroup; ++i)
    if (t >= g.tbegin[i]) a.w = g.w[i], a.ws = g.ws[i], a.out = g.out[i], a.n = g.n[i], first = g.tbegin[i];
  return t - first;
}

// ---------------------------------------------------------------- narrow
// Workgroup b owns output columns [16 NB b, 16 NB (b + 1)) and all M rows (MB
// 16-row blocks); NB is 1 but for groups whose 16-column tiles would take
// the CUs one and a half times.  (Below for NB = 1.)  Wave w sums ST = K / (128 S) of the 128-byte K chunks
// (the host guarantees K % (128 S) == 0): with S = 4 the contiguous slice
// w ST .. w ST + ST - 1, stage s reading chunk w ST + s; with S = 8 the
// waves interleave, stage s reading chunk ((s + b) mod ST) S + w, so that a
// workgroup's eight waves read eight consecutive chunks of every row and
// workgroups start at different chunks (down 4096 x 12288 at M = 2 / 8 / 16,
// graphs of 36 launches on MI355X: 10.90 / 10.93 / 11.98 us against 11.03 /
// 11.27 / 12.32 for contiguous slices; at K = 4096 with S = 4 the
// interleaved order was 0.4-0.8 us slower on qkv and o).  Each wave streams
// its chunks through its own ring of R stages: a stage holds 16 weight rows,
// then 16 MB activation
// rows, 128 bytes each; DMA instruction j fills rows 8j .. 8j + 7, lane l
// chunk l % 8 of row 8j + l / 8 with global chunk (l % 8) ^ (row % 8), so
// that the 16-row fragment reads (lane l: row l % 16) meet eight distinct
// bank groups.  Only the first LAL activation instructions are issued (the
// host picks LAL = ceil(M / 8)); lanes of rows >= M load nothing, so those
// LDS rows hold stale bytes whose products reach only accumulator rows >= M,
// which are never stored.  Weight rows past N re-read row N - 1.  A wave
// reads only its own ring, so the K loop needs no workgroup barrier: each
// stage is waited for with vmcnt (every issued instruction has a live lane,
// so the count is exact), and a slot is refilled only after the previous
// stage's fragment reads have returned.
template <int MB, int LAL, int S, int R, bool GROUP = false, int NB = 1>
__global__ __launch_bounds__(64 * S) void gemm_narrow(GemmArgs a, GroupArg<GROUP> group) {
  constexpr int ROWS = 16 * (NB + MB);
  constexpr int STAGE = ROWS * 128;
  constexpr int L = 2 * NB + LAL;  // DMA instructions per stage
  constexpr int RING = R * STAGE;
  static_assert(MB >= 1 && LAL >= 1 && LAL <= 2 * MB, "live activation loads");
  static_assert(R >= 2 && (R - 1) * L < 64, "ring depth");
  static_assert(S * RING <= 160 * 1024, "LDS");
  static_assert(S * MB * NB * 4 * 64 * (int)sizeof(int) <= S * RING, "the reduction reuses the rings");
  __shared__ __attribute__((aligned(1024))) int8_t lds[S * RING];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t n0 = own_tile(a, group, blockIdx.x) * 16 * NB;
  const uint32_t K = a.k, M = a.m, N = a.n;
  const uint32_t ST = K / (128 * S);
  int8_t* const ring = lds + wave * RING;

  const int8_t* src[L];
  bool live[L];
#pragma unroll
  for (int j = 0; j < L; ++j) {
    const int row = 8 * j + (lane >> 3);
    const size_t chunk = (size_t)(((lane & 7) ^ (row & 7)) * 16);
    if (row < 16 * NB) {
      const uint32_t g = n0 + row;
      src[j] = a.w + (size_t)(g < N ? g : N - 1) * K + chunk;
      live[j] = true;
    } else {
      const uint32_t g = (uint32_t)(row - 16 * NB);
      live[j] = g < M;
      src[j] = a.q + (size_t)(live[j] ? g : 0) * K + chunk;
    }
  }
  auto load = [&](uint32_t s) {
    int8_t* const base = ring + (s % R) * STAGE;
    const size_t kc = S >= 8 ? (size_t)((s + blockIdx.x) % ST) * S + wave : (size_t)wave * ST + s;
#pragma unroll
    for (int j = 0; j < L; ++j)
      if (live[j])
        __builtin_amdgcn_global_load_lds((const void*)(src[j] + kc * 128),
                                         W8A8_LDS_PTR(base + j * 1024 + lane * 16), 16, 0, 0);
  };

  const int fr = lane & 15, fq = lane >> 4;
  v4i acc[MB][NB];
#pragma unroll
  for (int t = 0; t < MB; ++t)
#pragma unroll
    for (int u = 0; u < NB; ++u) acc[t][u] = v4i{0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < R - 1; ++s)
    if ((uint32_t)s < ST) load(s);
  for (uint32_t s = 0; s < ST; ++s) {
    if (s + R - 1 < ST) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // stage s - 1's fragment reads returned
      load(s + R - 1);                                     // into stage s - 1's slot
      wait_vmcnt<(R - 1) * L>();                           // stage s landed
    } else {
      wait_vmcnt<0>();
    }
    const int8_t* const base = ring + (s % R) * STAGE;
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // the stage's two 64-byte k steps
      const int c = 4 * h + fq;
      v4i b[NB];
#pragma unroll
      for (int u = 0; u < NB; ++u) b[u] = *(const v4i*)(base + (16 * u + fr) * 128 + ((c ^ (fr & 7)) * 16));
#pragma unroll
      for (int t = 0; t < MB; ++t) {
        const int row = 16 * NB + 16 * t + fr;
        const v4i av = *(const v4i*)(base + row * 128 + ((c ^ (row & 7)) * 16));
#pragma unroll
        for (int u = 0; u < NB; ++u) acc[t][u] = mfma16(av, b[u], acc[t][u]);
      }
    }
  }
  __syncthreads();  // every wave is done with its ring
  int* const red = reinterpret_cast<int*>(lds);
#pragma unroll
  for (int t = 0; t < MB; ++t)
#pragma unroll
    for (int u = 0; u < NB; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[(((wave * MB + t) * NB + u) * 4 + v) * 64 + lane] = acc[t][u][v];
  __syncthreads();
  // value v of lane l of block (t, u): row 16 t + 4 (l / 16) + v, column
  // n0 + 16 u + l % 16
  for (int i = threadIdx.x; i < MB * NB * 4 * 64; i += 64 * S) {
    const int l = i & 63, v = (i >> 6) & 3, u = (i >> 8) % NB, t = (i >> 8) / NB;
    int sum = 0;
#pragma unroll
    for (int w = 0; w < S; ++w) sum += red[w * (MB * NB * 256) + i];
    const uint32_t r = 16 * t + 4 * (l >> 4) + v;
    const uint32_t c = n0 + 16 * u + (l & 15);
    if (r < M && c < N) epilogue_store(a, r, c, sum);
  }
}

// Epilogue of a wave's FM x FN grid of 32x32 accumulator blocks whose top
// left corner is (row0, col0).  Lane l, value v of block (i, j) is row
// row0 + 32i + 8(v / 4) + 4(l / 32) + v % 4, column col0 + 32j + l % 32.
// Every operand the epilogue reads (row scales, column scales, residuals)
// is loaded first, at clamped, always valid addresses, and every store comes
// after the last use of a load: stores count in the same in-order counter
// as loads, so a load issued after a store would wait for the store too.
//
// FULL: the whole grid of blocks lies inside the output, so nothing is clamped
// or guarded.  Every address is then a wave-uniform corner (scalar registers)
// plus one 32-bit lane offset, the same for all values: 4 (l / 32) rows and
// l % 32 columns (Off: 32 bits where the route keeps N at kMaxCols and below,
// so that its bytes fit).  Guarded values of one row of blocks take a per-lane
// product instead: between the guards' branches it is shorter than the scalar
// one (24576 x 4096 at M = 4 / 24 17.40 / 17.65 -> 17.28 / 17.50 us).
constexpr uint32_t kMaxCols = 1u << 26;
// Residuals of up to this many values per lane are loaded with the scales; a
// larger wave tile's, which the registers beside its accumulators do not hold,
// block by block, the next block's ahead of a block's stores.
constexpr int kResidualHeld = 64;

template <int EP, bool FULL, class Off, int FM, int FN>
__device__ __forceinline__ void store_blocks_as(const GemmArgs& a, const v16i (&acc)[FM][FN], uint32_t row0,
                                                uint32_t col0, int lane) {
  constexpr bool RES = EP == EP_F32_RES || EP == EP_BF16_RES;
  constexpr bool F32 = EP == EP_F32 || EP == EP_F32_RES;
  constexpr int ESZ = raw_i32(EP) || F32 ? 4 : 2;
  const uint32_t half = (uint32_t)lane >> 5, cl = (uint32_t)lane & 31;
  const Off lane_off = (Off)(4 * half) * a.n + cl;
  auto corner_row = [&](int i, int v) -> uint32_t { return row0 + 32 * i + (v >> 2) * 8 + (v & 3); };
  // byte address of value v of block (i, j) in an array of E-byte elements
  auto at = [&](const void* p, int i, int v, int j, auto esz) {
    constexpr uint32_t E = decltype(esz)::value;
    if constexpr (!FULL && FM == 1)
      return (char*)p + ((size_t)(corner_row(i, v) + 4 * half) * a.n + col0 + 32 * j + cl) * E;
    return (char*)p + ((size_t)corner_row(i, v) * a.n + col0 + 32 * j) * E + (size_t)(lane_off * E);
  };
  using E4 = std::integral_constant<uint32_t, 4>;
  using EO = std::integral_constant<uint32_t, ESZ>;
  auto inside = [&](int i, int v, int j) {
    return FULL || (corner_row(i, v) + 4 * half < a.m && col0 + 32 * j + cl < a.n);
  };
  if constexpr (raw_i32(EP)) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          if (inside(i, v, j)) {
            int32_t* const o = (int32_t*)at(a.out, i, v, j, EO{});
            if (EP == EP_SLAB) __builtin_nontemporal_store(acc[i][j][v], o);
            else *o = acc[i][j][v];
          }
    return;
  }
  constexpr int NB = FM * FN;  // block b: row block b % FM, column block b / FM
  constexpr bool HELD = NB * 16 <= kResidualHeld;
  constexpr int SLOTS = HELD ? NB : 2;
  float asc[FM][16], wsc[FN];
  float res[RES ? SLOTS : 1][16];
  auto load_res = [&](int b) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int i = b % FM, j = b / FM;
      res[b % SLOTS][v] =
          FULL ? *(const float*)at(a.residual, i, v, j, E4{})
               : a.residual[(size_t)min(corner_row(i, v) + 4 * half, a.m - 1) * a.n + min(col0 + 32 * j + cl, a.n - 1)];
    }
  };
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const uint32_t r = corner_row(i, v) + 4 * half;
      asc[i][v] = a.asc[FULL ? r : min(r, a.m - 1)];
    }
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const uint32_t c = col0 + 32 * j + cl;
    wsc[j] = a.ws[FULL ? c : min(c, a.n - 1)];
  }
  if constexpr (RES) {
#pragma unroll
    for (int b = 0; b < (HELD ? NB : 1); ++b) load_res(b);
  }
  // one wait for every load above, taken unconditionally: a wait first met
  // inside a guarded store would be repeated in each guarded store after it
  wait_vmcnt<0>();
  // The outputs are written non-temporally (no line of them is re-read by
  // this kernel).  Measured on MI355X, graphs of 16 distinct-weight launches
  // with random operands: o at M = 512 16.8 against 17.2-17.4 us, qkv
  // 22.5-22.7 against 23.0-23.3, gate_up at M = 129 30.9 against 31.2-31.4.
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int i = b % FM, j = b / FM;
    if constexpr (RES && !HELD) {
      __builtin_amdgcn_sched_barrier(0);
      if (b + 1 < NB) load_res(b + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float val = dequant(acc[i][j][v], asc[i][v], wsc[j]);
      const float cmb = RES ? bf16_rne(res[RES ? b % SLOTS : 0][v] + val) : 0.f;
      if (!inside(i, v, j)) continue;
      if constexpr (F32) {
        if (a.out) __builtin_nontemporal_store(val, (float*)at(a.out, i, v, j, EO{}));
        if (RES) *(float*)at(a.combined, i, v, j, EO{}) = cmb;
      } else {
        if (a.out)
          __builtin_nontemporal_store((uint16_t)(__float_as_uint(val) >> 16), (uint16_t*)at(a.out, i, v, j, EO{}));
        if (RES) *(uint16_t*)at(a.combined, i, v, j, EO{}) = (uint16_t)(__float_as_uint(cmb) >> 16);
      }
    }
  }
}

template <int EP, class Off = uint32_t, int FM, int FN>
__device__ __forceinline__ void store_blocks(const GemmArgs& a, const v16i (&acc)[FM][FN], uint32_t row0,
                                             uint32_t col0, int lane) {
  if ((size_t)row0 + 32 * FM <= a.m && (size_t)col0 + 32 * FN <= a.n)
    store_blocks_as<EP, true, Off, FM, FN>(a, acc, row0, col0, lane);
  else
    store_blocks_as<EP, false, Off, FM, FN>(a, acc, row0, col0, lane);
}

// Prefill GEMM.  Workgroup = 8 waves (two per SIMD: while one wave waits on
// LDS the other keeps the matrix core busy), output tile BM x BN, wave tile
// WM x WN built from 32x32 MFMA blocks.  K advances in 128-byte stages, so
// every DMA row request is one whole 128-byte cache line.
//
// LDS holds two rings: activations (A, BM rows of 128 bytes per stage, SA
// slots) and weights (B, BN rows, SB >= SA slots).  Weight lines mostly miss
// L2, so they can be requested further ahead than the activation lines,
// which every workgroup shares.  Batch(kt) = {A(kt + SA - 1), B(kt + SB - 1)}
// is issued during stage kt (A first) into the slots stage kt - 1 released.
// Loads complete in issue order, so at the end of stage kt "A(kt + 1) and
// B(kt + 1) have landed" means: at most the loads issued after A(kt + 1)
// remain -- the B half of its batch when SB > SA (when SB == SA that half is
// B(kt + 1) itself and must land too), plus the SA - 2 whole batches after
// it.
//
// 16-byte chunk c of LDS row r sits at chunk c ^ ((r >> 1) & 7): sixteen
// consecutive rows (two per 256-byte bank window) of one fragment read then
// hit sixteen different 16-byte bank groups.  Sub-step i of a stage covers
// k bytes [32i, 32i + 32): lane l (row / column l % 32, half h = l / 32)
// reads chunk 2i + h -- the same lane -> k map for A and B.
// Tiles are numbered XCD-aware (each XCD a contiguous run) and, within that,
// in strips of kStrip M tiles that walk all N tiles, so that the 32 tiles an
// XCD runs at once are about 4 x 8: they share 4 activation and 8 weight
// panels through its L2 while they advance through K together.  M fastest over
// all M tiles instead, with each tile starting K at its own stage, fetched
// most panels once per tile: 24576 x 4096 at M = 4096, f32, 256 x 192 tiles
// 484 -> 443 us; strips of 4 / 8 / 16 on 256 x 256 tiles 387 / 397 / 430.
constexpr uint32_t kStrip = 4;
// Rotated K: in a launch of one round over one column of tiles (unsplit, K % 128
// == 0, eight waves), stage kt of tile t reads K chunk (kt + t) mod KT; the i32 sums
// are exact in any order.  Every workgroup walks the same weights there, and in
// step all rows of a stage can lie on one memory channel: 64 x 16384 at M = 22,000
// 87 -> 69 us.  With more columns the panels shared in step are worth as much:
// rotated / in order with distinct weights, BF16, 6144 x 4096 at M = 129 14.9 /
// 13.9, M = 256 16.2 / 16.6, M = 512 21.6 / 21.9, M = 2048 56.8 / 51.8; 6144 x 8192 at
// M = 256 30.0 / 29.1, 6144 x 2048 10.1 / 10.0; 4096 x 4096 at M = 4096 69 / 66.
constexpr uint64_t kCus = 256;
constexpr uint32_t kMaxK = 1u << 23;  // 256 rows of K bytes stay within a 32-bit offset

// TAIL (K % 128 != 0, any N): the last stage is partial.  A lane whose 16-byte
// chunk lies past K reads zeros for the activation row, and its weight row's
// first chunk (any bytes: their products are zero), so nothing outside the
// operands is read and the sums are exact.  These launches take four waves
// per workgroup (NW), as does the 64 x 64 tile; two workgroups share a CU where the
// rings take 80 KiB.
__device__ const v4i kZeroChunk = {0, 0, 0, 0};

constexpr int waves_per_simd(int nw, int lds_bytes) { return nw == 8 || lds_bytes <= 80 * 1024 ? 2 : 1; }

template <int BM, int BN, int WM, int WN, int SA, int SB, int EP, bool GROUP = false, int NW = 8, bool TAIL = false>
__global__ __launch_bounds__(64 * NW, (waves_per_simd(NW, (SA * BM + SB * BN) * 128))) void gemm_dma(
    GemmArgs a, uint32_t tiles_m, uint32_t tiles_n, uint32_t splits, GroupArg<GROUP> group) {
  constexpr int WAVES_N = BN / WN;
  static_assert((BM / WM) * (BN / WN) == NW, "one wave tile per wave");
  static_assert(WM % 32 == 0 && WN % 32 == 0 && BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "tile shape");
  static_assert(SA >= 2 && SB >= SA && SB >= 3 && SB <= 8, "ring depths");
  constexpr int FM = WM / 32, FN = WN / 32;
  constexpr int LA = BM / 8 / NW, LB = BN / 8 / NW;  // DMA loads (8 rows x 128 B) per wave per stage
  constexpr int L = LA + LB;
  constexpr int ASL = BM * 128, BSL = BN * 128;
  static_assert(SA * ASL + SB * BSL <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024))) int8_t lds[SA * ASL + SB * BSL];
  int8_t* const ldsA = lds;
  int8_t* const ldsB = lds + SA * ASL;

  // Split-K (splits > 1, EP_SLAB or EP_I32): workgroup (tile, split) sums K range
  // [split * K / splits, (split + 1) * K / splits) into i32 slab `split` of
  // a.out; a separate epilogue kernel adds the slabs (exact) and dequantizes.
  const uint32_t T = tiles_m * tiles_n, G = T * splits;
  uint32_t Lt = blockIdx.x;
  if (G % 8 == 0) Lt = (blockIdx.x % 8) * (G / 8) + blockIdx.x / 8;
  const uint32_t split = Lt / T;
  Lt %= T;
  const uint32_t strip = kStrip * (T / tiles_m), s0 = Lt / strip * kStrip, in = Lt % strip;
  const uint32_t sm = min(kStrip, tiles_m - s0);  // M tiles of this strip
  const uint32_t m0 = (s0 + in % sm) * BM, n0 = own_tile(a, group, in / sm) * BN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wm0 = (wave / WAVES_N) * WM, wn0 = (wave % WAVES_N) * WN;
  const uint32_t K = a.k, KT = TAIL ? K / 128 + 1 : K / 128 / splits;
  const size_t kbase = (size_t)split * KT * 128;
  if (raw_i32(EP)) a.out = reinterpret_cast<int32_t*>(a.out) + (size_t)split * a.m * a.n;
  const bool turned = splits == 1 && tiles_n == 1 && T <= kCus;
  const uint32_t rot = !TAIL && NW == 8 && turned ? Lt % KT : 0;
  auto kc = [&](uint32_t kt) -> size_t {  // byte offset of stage kt
    if constexpr (TAIL || NW != 8) return (size_t)kt * 128;
    const uint32_t c = kt + rot;
    return (size_t)(c >= KT ? c - KT : c) * 128;
  };

  // Sources of this wave's DMA loads (8 rows each); rows past M / N re-read
  // the tile's first row (their products only reach accumulator cells that are never
  // stored).  Lane l fills LDS chunk l % 8 of row l / 8 with global chunk
  // (l % 8) ^ key(row).
  // An address is the tile's first row (scalar registers) plus a 32-bit lane
  // offset (the routes keep K at kMaxK and below).
  using Off = std::conditional_t<TAIL, size_t, uint32_t>;
  const int8_t* const srcA = a.q + (size_t)m0 * K + kbase;
  const int8_t* const srcB = a.w + (size_t)n0 * K + kbase;
  auto lds_row = [&](int g) { return (uint32_t)(8 * g + (lane >> 3)); };  // row group g of 8 rows
  auto chunk = [&](int g) { return (uint32_t)((lane & 7) ^ ((lds_row(g) >> 1) & 7)) * 16; };
  Off offA[LA], offB[LB];
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const uint32_t row = lds_row(wave * LA + j);
    offA[j] = (Off)(m0 + row < a.m ? row : 0) * K + (TAIL ? 0 : chunk(wave * LA + j));
  }
#pragma unroll
  for (int j = 0; j < LB; ++j) {
    const uint32_t row = lds_row(wave * LB + j);
    offB[j] = (Off)(n0 + row < a.n ? row : 0) * K + (TAIL ? 0 : chunk(wave * LB + j));
  }
  auto loadA = [&](uint32_t kt, int j) {
    const int8_t* p = srcA + kc(kt) + offA[j];
    if constexpr (TAIL) {
      const uint32_t kk = kt * 128 + chunk(wave * LA + j);
      p = kk < K ? srcA + offA[j] + kk : reinterpret_cast<const int8_t*>(&kZeroChunk);
    }
    __builtin_amdgcn_global_load_lds((const void*)p,
                                     W8A8_LDS_PTR(ldsA + (kt % SA) * ASL + (wave * LA + j) * 1024 + lane * 16),
                                     16, 0, 0);
  };
  auto loadB = [&](uint32_t kt, int j) {
    const int8_t* p = srcB + kc(kt) + offB[j];
    if constexpr (TAIL) {
      const uint32_t kk = kt * 128 + chunk(wave * LB + j);
      p = srcB + offB[j] + (kk < K ? kk : 0);
    }
    __builtin_amdgcn_global_load_lds((const void*)p,
                                     W8A8_LDS_PTR(ldsB + (kt % SB) * BSL + (wave * LB + j) * 1024 + lane * 16),
                                     16, 0, 0);
  };
  const int fr = lane & 31, fh = lane >> 5;
  int off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) off[i] = fr * 128 + (((2 * i + fh) ^ ((fr >> 1) & 7)) * 16);
  v16i acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = v16i{};
  auto rd = [&](uint32_t kt, int i, v4i (&af)[FM], v4i (&bf)[FN]) {
    const int8_t* ba = ldsA + (kt % SA) * ASL;
    const int8_t* bb = ldsB + (kt % SB) * BSL;
#pragma unroll
    for (int f = 0; f < FM; ++f) af[f] = *(const v4i*)(ba + (wm0 + 32 * f) * 128 + off[i]);
#pragma unroll
    for (int j = 0; j < FN; ++j) bf[j] = *(const v4i*)(bb + (wn0 + 32 * j) * 128 + off[i]);
  };
  auto mm = [&](const v4i (&af)[FM], const v4i (&bf)[FN]) {
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[f][j] = mfma32(af[f], bf[j], acc[f][j]);
  };
  // The same MFMAs with the loads load(0) .. load(N - 1) issued evenly between
  // them, and kept there: the wave's MFMAs do not queue behind a burst of DMA
  // issues after the barrier.
  auto mm_load = [&](const v4i (&af)[FM], const v4i (&bf)[FN], auto n, auto load) {
    constexpr int N = decltype(n)::value, MF = FM * FN;
#pragma unroll
    for (int i = 0; i < MF; ++i) {
      acc[i / FN][i % FN] = mfma32(af[i / FN], bf[i % FN], acc[i / FN][i % FN]);
      const int lo = (i * N + MF - 1) / MF, hi = ((i + 1) * N + MF - 1) / MF;
      if (lo == hi) continue;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < N; ++j)
        if (j >= lo && j < hi) load(j);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using LoadsA = std::integral_constant<int, LA>;
  using LoadsB = std::integral_constant<int, LB>;

  // Prologue: stages 0 .. SB - 2 (A only up to SA - 2), stage by stage, A
  // before B; then wait for stage 0.
#pragma unroll
  for (int s = 0; s < SB - 1; ++s) {
    if (s >= (int)KT) break;
    if (s < SA - 1)
#pragma unroll
      for (int j = 0; j < LA; ++j) loadA(s, j);
#pragma unroll
    for (int j = 0; j < LB; ++j) loadB(s, j);
  }
  if (KT >= (uint32_t)SB - 1) wait_vmcnt<(SA - 2) * LA + (SB - 2) * LB>();
  else wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();
  v4i a0[FM], b0[FN], a1[FM], b1[FN];
  if (SA - 1 < KT)
#pragma unroll
    for (int j = 0; j < LA; ++j) loadA(SA - 1, j);
  rd(0, 0, a0, b0);
  // Fragments of the next sub-step are read while the current one's MFMAs
  // run.  The loop body has no branch between a read and its use, so the
  // compiler's LDS waits keep the newest reads in flight.  Batch(kt) goes out
  // among the MFMAs of two sub-steps: A(kt + SA - 1) with the last ones of
  // stage kt - 1 (after the barrier that released its slot), B(kt + SB - 1)
  // with the first ones of stage kt.
  auto stage = [&](uint32_t kt, auto all) {
    constexpr bool ALL = decltype(all)::value;  // every load of this stage exists
    const bool more_b = ALL || kt + SB - 1 < KT, more_a = ALL || kt + SA < KT;
    rd(kt, 1, a1, b1);
    mm_load(a0, b0, LoadsB{}, [&](int j) { if (more_b) loadB(kt + SB - 1, j); });
    rd(kt, 2, a0, b0);
    mm(a1, b1);
    rd(kt, 3, a1, b1);
    mm(a0, b0);
    // A(kt + 1), B(kt + 1) landed (every load counted here exists while batch
    // kt was complete)
    if (more_b) wait_vmcnt<(SB > SA ? LB : 0) + (SA - 2) * L>();
    else wait_vmcnt<0>();
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's reads of stage kt returned
    __builtin_amdgcn_s_barrier();         // all waves: stage kt + 1 landed, stage kt read
    rd(kt + 1, 0, a0, b0);
    mm_load(a1, b1, LoadsA{}, [&](int j) { if (more_a) loadA(kt + SA, j); });
  };
  uint32_t kt = 0;
  constexpr uint32_t AHEAD = SB > SA ? SB - 1 : SA;
  for (; kt + AHEAD < KT; ++kt) stage(kt, std::true_type{});
  for (; kt + 1 < KT; ++kt) stage(kt, std::false_type{});
  rd(KT - 1, 1, a1, b1);
  mm(a0, b0);
  rd(KT - 1, 2, a0, b0);
  mm(a1, b1);
  rd(KT - 1, 3, a1, b1);
  mm(a0, b0);
  mm(a1, b1);

  store_blocks<EP, Off>(a, acc, m0 + wm0, n0 + wn0, lane);
}

// A 128 x 128 wave tile's accumulators leave no registers for residuals.
template <int WM, int WN>
constexpr bool kResidualTile = WM * WN < 128 * 128;

template <int BM, int BN, int WM, int WN, int SA, int SB, int NW = 8, bool TAIL = false>
static hipError_t launch_dma(hipStream_t st, const GemmArgs& a) {
  const uint32_t tm = (a.m + BM - 1) / BM, tn = (a.n + BN - 1) / BN;
  auto k = a.out_dtype == W8A8_OUT_I32   ? gemm_dma<BM, BN, WM, WN, SA, SB, EP_I32, false, NW, TAIL>
           : a.out_dtype == W8A8_OUT_F32 ? gemm_dma<BM, BN, WM, WN, SA, SB, EP_F32, false, NW, TAIL>
                                         : gemm_dma<BM, BN, WM, WN, SA, SB, EP_BF16, false, NW, TAIL>;
  if (a.residual) {
    if constexpr (kResidualTile<WM, WN>)
      k = a.out_dtype == W8A8_OUT_F32 ? gemm_dma<BM, BN, WM, WN, SA, SB, EP_F32_RES, false, NW, TAIL>
                                      : gemm_dma<BM, BN, WM, WN, SA, SB, EP_BF16_RES, false, NW, TAIL>;
    else
      return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL(k, dim3(tm * tn), dim3(64 * NW), 0, st, a, tm, tn, 1u, NoGroup{});
  return hipGetLastError();
}

// Cache policy of a load streamed once (the weights of a single M tile): the
// non-temporal bit, so the lines do not displace the activations that every
// workgroup re-reads from L2.
constexpr int kCpolNT = 2;

// s_waitcnt vmcnt(n) for a wave-uniform n known only at run time (n <= 20).
__device__ __forceinline__ void wait_vmcnt_dyn(int n) {
  switch (n) {
    case 0: wait_vmcnt<0>(); break;
    case 1: wait_vmcnt<1>(); break;
    case 2: wait_vmcnt<2>(); break;
    case 3: wait_vmcnt<3>(); break;
    case 4: wait_vmcnt<4>(); break;
    case 5: wait_vmcnt<5>(); break;
    case 6: wait_vmcnt<6>(); break;
    case 7: wait_vmcnt<7>(); break;
    case 8: wait_vmcnt<8>(); break;
    case 9: wait_vmcnt<9>(); break;
    case 10: wait_vmcnt<10>(); break;
    case 11: wait_vmcnt<11>(); break;
    case 12: wait_vmcnt<12>(); break;
    case 13: wait_vmcnt<13>(); break;
    case 14: wait_vmcnt<14>(); break;
    case 15: wait_vmcnt<15>(); break;
    case 16: wait_vmcnt<16>(); break;
    case 17: wait_vmcnt<17>(); break;
    case 18: wait_vmcnt<18>(); break;
    case 19: wait_vmcnt<19>(); break;
    default: wait_vmcnt<20>(); break;
  }
}

// Prefill / small-batch GEMM for M <= MA (gemm_tall, MA = 64, 160 or 256).  One M tile
// of MA rows holds every activation row, so each weight tile is read from
// HBM once, and no DMA or MFMA goes to a second M tile holding a few rows.
// MA = 160 and 256: the eight waves are stacked along M (wave w: rows
// 32w .. 32w + 31, all BN columns), so a wave reads one activation fragment
// per k step for its BN / 32 MFMAs.  MA = 64 (M <= 64, one or two 32-row
// blocks): the 32 x 32 output blocks are dealt to the waves one each (block
// b = row block * BN / 32 + column block goes to wave b), so the SIMDs (wave
// w runs on SIMD w % 4) share the MFMAs instead of one or two waves holding
// them all.  Measured on MI355X, graphs of 16 distinct-weight launches with
// random operands, rows-per-wave -> one block per wave: at M = 16 qkv 11.7
// -> 10.6 us, o 9.3 -> 8.6, gate_up 21.0-21.4 -> 18.1, down 15.6 -> 13.8;
// at M = 64 qkv 13.0 -> 12.0, o 10.9 -> 10.4, gate_up 22.1-23.3 -> 20.0-20.4,
// down 17.6-18.2 -> 16.3.  With more row blocks the same dealing reads twice
// the LDS fragment bytes per MFMA for no better balance (M = 129: level;
// M = 200: gate_up 33.0 -> 37.8), so those tiles keep rows per wave.
// A wave that holds no block only moves data.
//
// Rings as in gemm_dma: activations (SA slots of MA rows; the lines are
// shared by every workgroup and come from L2 or MALL) and weights (SB slots;
// the lines come from HBM and are read once, non-temporal).  With few MFMAs
// per stage the stage is short, so both rings look several stages ahead.
// Loads complete in issue order, so a weight load issued before an
// activation load has to land before that activation's wait: weight slots
// beyond the activation ring's depth add no lookahead, and most plans use
// equal depths.
//
// A stage's DMA instructions (8 rows x 128 bytes each) are dealt to the
// waves round-robin, separately for the ceil(M / 8) activation row groups --
// rows past the last group are never loaded -- and the BN / 8 weight row
// groups, so a wave issues na activation and nb weight instructions per stage
// and counts its waits with its own na, nb.  During stage kt it issues
// A(kt + SA - 1), then B(kt + SB - 1).
// Split-K as in gemm_dma: workgroup (tile, split) writes i32 slab `split`.
// ROT (unsplit launches): each workgroup starts K at its own stage (stage kt
// reads K chunk (kt + tile) mod KT; the i32 sums are exact in any order), so
// that the workgroups do not all read the same 128-byte column of their
// weight rows at once.  Measured on MI355X (graphs of 16 distinct-weight
// launches): gate_up 24576 x 4096 at M = 64 22.2 against 25.1 us, M = 129
// 29.4-29.7 against 30.3-31.4, M = 193 32.8 against 34.5-35.0.  Split-K
// launches, whose slabs already start at different K offsets, measured level
// or up to 1.3% slower rotated, and keep the order.
// TIMED (diagnostics only, w8a8_diag_gemm_timeline): every wave also
// records the 100 MHz device clock at its start, once stage 0 has landed
// (the prologue), after its last MFMA / DMA issue, and once its stores are
// acknowledged, into stamps[4 g .. 4 g + 3] (g = workgroup * 8 + wave).
constexpr bool kRotateK = true;

template <int BN, int SA, int SB, int MA, int EP, bool ROT = false, bool TIMED = false, bool GROUP = false>
__global__ __launch_bounds__(512) void gemm_tall(GemmArgs a, uint32_t tiles_n, uint32_t splits,
                                                 uint64_t* stamps, GroupArg<GROUP> group) {
  uint64_t ts[4] = {0, 0, 0, 0};
  if constexpr (TIMED) ts[0] = __builtin_amdgcn_s_memrealtime();
  constexpr int FN = BN / 32;
  constexpr int ASL = MA * 128, BSL = BN * 128;
  constexpr uint32_t NB = BN / 8;
  constexpr int kMaxA = (MA / 8 + 7) / 8, kMaxB = (NB + 7) / 8;
  static_assert(BN % 32 == 0 && BN <= 128 && MA % 32 == 0 && MA <= 256, "tile");
  static_assert(SA >= 2 && SB >= SA && SA * ASL + SB * BSL <= 160 * 1024, "LDS");
  static_assert((SB > SA ? kMaxB : 0) + (SA - 2) * (kMaxA + kMaxB) <= 20 &&
                    (SA - 2) * kMaxA + (SB - 2) * kMaxB <= 20,
                "wait range");
  __shared__ __attribute__((aligned(1024))) int8_t lds[SA * ASL + SB * BSL];
  int8_t* const ldsA = lds;
  int8_t* const ldsB = lds + SA * ASL;

  const uint32_t G = tiles_n * splits;
  uint32_t Lt = blockIdx.x;
  if (G % 8 == 0) Lt = (blockIdx.x % 8) * (G / 8) + blockIdx.x / 8;
  const uint32_t split = Lt / tiles_n;
  const uint32_t n0 = own_tile(a, group, Lt % tiles_n) * BN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t K = a.k, KT = K / 128 / splits;
  const size_t kbase = (size_t)split * KT * 128;
  if (raw_i32(EP)) a.out = reinterpret_cast<int32_t*>(a.out) + (size_t)split * a.m * a.n;

  // This wave's DMA instructions: activation row groups w, w + 8, ... below
  // ceil(M / 8), weight row groups w, w + 8, ... below BN / 8.  Lane l fills
  // LDS chunk l % 8 of row l / 8 with global chunk (l % 8) ^ key(row).
  const uint32_t NA = (a.m + 7) / 8;
  const int na = (int)((NA + 7 - (uint32_t)wave) / 8);
  const int nb = (int)((NB + 7 - (uint32_t)wave) / 8);
  const int8_t* srcA[kMaxA];
  const int8_t* srcB[kMaxB];
#pragma unroll
  for (int j = 0; j < kMaxA; ++j) {
    const uint32_t row = 8 * (wave + 8 * j) + (lane >> 3);
    srcA[j] = a.q + (size_t)min(row, a.m - 1) * K + kbase + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
  }
#pragma unroll
  for (int j = 0; j < kMaxB; ++j) {
    const uint32_t br = 8 * (wave + 8 * j) + (lane >> 3);  // row within the weight tile
    srcB[j] = a.w + (size_t)min(n0 + br, a.n - 1) * K + kbase + ((lane & 7) ^ ((br >> 1) & 7)) * 16;
  }
  // ROT: stage kt reads global K chunk (kt + rot) mod KT, rot = Lt mod KT, so
  // the workgroups do not all read the same 128-byte column of their weight
  // rows at once.
  const uint32_t rot = ROT ? Lt % KT : 0;
  auto kc = [&](uint32_t kt) -> size_t {
    const uint32_t c = kt + rot;
    return (size_t)(c >= KT ? c - KT : c) * 128;
  };
  auto issueA = [&](uint32_t kt) {
#pragma unroll
    for (int j = 0; j < kMaxA; ++j)
      if (j < na)
        __builtin_amdgcn_global_load_lds((const void*)(srcA[j] + kc(kt)),
                                         W8A8_LDS_PTR(ldsA + (kt % SA) * ASL + 1024 * (wave + 8 * j) + lane * 16),
                                         16, 0, 0);
  };
  auto issueB = [&](uint32_t kt) {
#pragma unroll
    for (int j = 0; j < kMaxB; ++j)
      if (j < nb)
        __builtin_amdgcn_global_load_lds((const void*)(srcB[j] + kc(kt)),
                                         W8A8_LDS_PTR(ldsB + (kt % SB) * BSL + 1024 * (wave + 8 * j) + lane * 16),
                                         16, 0, kCpolNT);
  };
  auto batch = [&](uint32_t kt) {
    if (kt + SA - 1 < KT) issueA(kt + SA - 1);
    if (kt + SB - 1 < KT) issueB(kt + SB - 1);
  };
  // end of stage kt: A(kt + 1) and B(kt + 1) landed; in flight may remain the
  // B half of A(kt + 1)'s batch (when SB > SA) and the SA - 2 whole batches
  // after it
  auto wait_next = [&](uint32_t kt) {
    if (kt + SB - 1 < KT) wait_vmcnt_dyn((SB > SA ? nb : 0) + (SA - 2) * (na + nb));
    else wait_vmcnt<0>();
  };

  const int fr = lane & 31, fh = lane >> 5;
  int off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) off[i] = fr * 128 + (((2 * i + fh) ^ ((fr >> 1) & 7)) * 16);
  // Stage pipeline shared by both mappings: fragments of sub-step i + 1 are
  // read while the MFMAs of sub-step i issue.  rd(kt, i, f) reads sub-step i
  // of stage kt into f; mm(f) issues its MFMAs.
  auto pipeline = [&](auto& f0, auto& f1, auto rd, auto mm) {
    batch(0);
    rd(0, 0, f0);
    for (uint32_t kt = 0; kt + 1 < KT; ++kt) {
      rd(kt, 1, f1);
      mm(f0);
      rd(kt, 2, f0);
      mm(f1);
      rd(kt, 3, f1);
      mm(f0);
      wait_next(kt);
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's reads of stage kt returned
      __builtin_amdgcn_s_barrier();
      batch(kt + 1);
      rd(kt + 1, 0, f0);
      mm(f1);
    }
    rd(KT - 1, 1, f1);
    mm(f0);
    rd(KT - 1, 2, f0);
    mm(f1);
    rd(KT - 1, 3, f1);
    mm(f0);
    mm(f1);
  };
  // rows past M, or no block: this wave only moves its share of the data
  auto move_only = [&]() {
    batch(0);
    for (uint32_t kt = 0; kt + 1 < KT; ++kt) {
      wait_next(kt);
      __builtin_amdgcn_s_barrier();
      batch(kt + 1);
    }
  };

  // Prologue: stages 0 .. SB - 2 (activations up to SA - 2), stage by stage;
  // then wait for A(0) and B(0).
  for (int s = 0; s < SB - 1; ++s) {
    if (s >= (int)KT) break;
    if (s < SA - 1) issueA(s);
    issueB(s);
  }
  if (KT >= (uint32_t)SB - 1) wait_vmcnt_dyn((SA - 2) * na + (SB - 2) * nb);
  else wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();
  if constexpr (TIMED) ts[1] = __builtin_amdgcn_s_memrealtime();
  auto stamp_stream_end = [&]() {
    if constexpr (TIMED) ts[2] = __builtin_amdgcn_s_memrealtime();
  };

  if constexpr (MA == 64) {
    // one 32 x 32 block per wave: block `wave` of the (M / 32) x FN grid
    const uint32_t T = (a.m + 31) / 32 * FN;
    static_assert(2 * FN <= 8, "one block per wave");
    if ((uint32_t)wave < T) {
      const uint32_t mb = (uint32_t)wave / FN, nbk = (uint32_t)wave % FN;
      const int8_t* const aa = ldsA + mb * 32 * 128;
      const int8_t* const bb = ldsB + nbk * 32 * 128;
      struct Frag { v4i a, b; };
      v16i acc = v16i{};
      Frag f0, f1;
      pipeline(f0, f1,
               [&](uint32_t kt, int i, Frag& f) {
                 f.a = *(const v4i*)(aa + (kt % SA) * ASL + off[i]);
                 f.b = *(const v4i*)(bb + (kt % SB) * BSL + off[i]);
               },
               [&](const Frag& f) { acc = mfma32(f.a, f.b, acc); });
      stamp_stream_end();
      const v16i blocks[1][1] = {{acc}};
      store_blocks<EP>(a, blocks, 32 * mb, n0 + 32 * nbk, lane);
    } else {
      move_only();
      stamp_stream_end();
    }
  } else {
    if (32u * wave < a.m) {
      struct Frag { v4i a, b[FN]; };
      v16i acc[FN];
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[j] = v16i{};
      Frag f0, f1;
      pipeline(f0, f1,
               [&](uint32_t kt, int i, Frag& f) {
                 f.a = *(const v4i*)(ldsA + (kt % SA) * ASL + (32 * wave) * 128 + off[i]);
                 const int8_t* bb = ldsB + (kt % SB) * BSL;
#pragma unroll
                 for (int j = 0; j < FN; ++j) f.b[j] = *(const v4i*)(bb + (32 * j) * 128 + off[i]);
               },
               [&](const Frag& f) {
#pragma unroll
                 for (int j = 0; j < FN; ++j) acc[j] = mfma32(f.a, f.b[j], acc[j]);
               });
      stamp_stream_end();
      const v16i (&blocks)[1][FN] = *reinterpret_cast<const v16i(*)[1][FN]>(&acc);
      store_blocks<EP>(a, blocks, 32 * wave, n0, lane);
    } else {
      move_only();
      stamp_stream_end();
    }
  }
  if constexpr (TIMED) {
    __builtin_amdgcn_s_waitcnt(0);
    ts[3] = __builtin_amdgcn_s_memrealtime();
    if (lane == 0) {
      uint64_t* o = stamps + ((size_t)blockIdx.x * 8 + wave) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = ts[i];
    }
  }
}

constexpr uint32_t kMaxSplits = 4;  // split-K plans use 2 or 4 slabs

// A slab quad; NT: the slabs were streamed (EP_SLAB) and are read once.
template <bool NT>
__device__ __forceinline__ v4i load_slab(const int32_t* p) {
  if (NT) return __builtin_nontemporal_load(reinterpret_cast<const v4i*>(p));
  return *reinterpret_cast<const v4i*>(p);
}

// Split-K epilogue: out[r][c] = epilogue(sum over slabs of partials[s][r][c]).
// The i32 sum is exact in any order.  blockIdx.y walks rows (the row scale is
// one scalar load), each thread four consecutive columns (n % 4 == 0), so the
// slab, weight-scale and residual loads are all issued up front.
template <int EP, bool NT>
__global__ __launch_bounds__(256) void splitk_epilogue(GemmArgs a, const int32_t* __restrict__ partials,
                                                        uint32_t splits) {
  constexpr bool RES = EP == EP_F32_RES || EP == EP_BF16_RES;
  const size_t mn = (size_t)a.m * a.n;
  const uint32_t c = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (c >= a.n) return;
  float wsc[4] = {0.f, 0.f, 0.f, 0.f};
  if (EP != EP_I32)
#pragma unroll
    for (int j = 0; j < 4; ++j) wsc[j] = a.ws[c + j];
  for (uint32_t r = blockIdx.y; r < a.m; r += gridDim.y) {
    const size_t i = (size_t)r * a.n + c;
    // every operand of the row first -- up to kMaxSplits slabs (slab index
    // clamped, surplus slabs masked), the row scale, the residuals -- so one
    // load round trip covers them; the stores come last
    v4i part[kMaxSplits];
#pragma unroll
    for (uint32_t s = 0; s < kMaxSplits; ++s)
      part[s] = load_slab<NT>(partials + min(s, splits - 1) * mn + i);
    const float asc = EP != EP_I32 ? a.asc[r] : 0.f;
    float res[4] = {0.f, 0.f, 0.f, 0.f};
    if (RES)
#pragma unroll
      for (int j = 0; j < 4; ++j) res[j] = a.residual[i + j];
    v4i acc = part[0];
#pragma unroll
    for (uint32_t s = 1; s < kMaxSplits; ++s)
      if (s < splits) acc += part[s];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const size_t o = i + j;
      if (EP == EP_I32) {
        reinterpret_cast<int32_t*>(a.out)[o] = acc[j];
        continue;
      }
      const float v = dequant(acc[j], asc, wsc[j]);
      if (EP == EP_F32 || EP == EP_F32_RES) {
        if (a.out) reinterpret_cast<float*>(a.out)[o] = v;
        if (RES) reinterpret_cast<float*>(a.combined)[o] = bf16_rne(res[j] + v);
      } else {
        if (a.out) reinterpret_cast<uint16_t*>(a.out)[o] = (uint16_t)(__float_as_uint(v) >> 16);
        if (RES)
          reinterpret_cast<uint16_t*>(a.combined)[o] = (uint16_t)(__float_as_uint(bf16_rne(res[j] + v)) >> 16);
      }
    }
  }
}

// The same epilogue with 8 columns per thread, for n % 8 == 0 and 16-byte
// aligned scales, residuals and outputs: every operand moves in 16-byte
// loads and stores (one store of 8 BF16 values), so a row costs a quarter of
// the 4-column kernel's store instructions.
template <int EP, bool NT>
__global__ __launch_bounds__(256) void splitk_epilogue8(GemmArgs a, const int32_t* __restrict__ partials,
                                                         uint32_t splits) {
  constexpr bool RES = EP == EP_F32_RES || EP == EP_BF16_RES;
  constexpr bool F32 = EP == EP_F32 || EP == EP_F32_RES;
  const size_t mn = (size_t)a.m * a.n;
  const uint32_t c = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (c >= a.n) return;
  float wsc[8] = {};
  if (EP != EP_I32) {
    const v4i w0 = *reinterpret_cast<const v4i*>(a.ws + c), w1 = *reinterpret_cast<const v4i*>(a.ws + c + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      wsc[j] = __int_as_float(w0[j]);
      wsc[4 + j] = __int_as_float(w1[j]);
    }
  }
  for (uint32_t r = blockIdx.y; r < a.m; r += gridDim.y) {
    const size_t i = (size_t)r * a.n + c;
    // every operand of the row first (slab index clamped, surplus slabs
    // masked), the stores last
    v4i p0[kMaxSplits], p1[kMaxSplits];
#pragma unroll
    for (uint32_t s = 0; s < kMaxSplits; ++s) {
      const int32_t* ps = partials + min(s, splits - 1) * mn + i;
      p0[s] = load_slab<NT>(ps);
      p1[s] = load_slab<NT>(ps + 4);
    }
    const float asc = EP != EP_I32 ? a.asc[r] : 0.f;
    v4i r0 = {0, 0, 0, 0}, r1 = {0, 0, 0, 0};
    if (RES) {
      r0 = *reinterpret_cast<const v4i*>(a.residual + i);
      r1 = *reinterpret_cast<const v4i*>(a.residual + i + 4);
    }
    v4i s0 = p0[0], s1 = p1[0];
#pragma unroll
    for (uint32_t s = 1; s < kMaxSplits; ++s)
      if (s < splits) {
        s0 += p0[s];
        s1 += p1[s];
      }
    if (EP == EP_I32) {
      int32_t* o = reinterpret_cast<int32_t*>(a.out) + i;
      *reinterpret_cast<v4i*>(o) = s0;
      *reinterpret_cast<v4i*>(o + 4) = s1;
      continue;
    }
    float v[8], cmb[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = dequant(j < 4 ? s0[j] : s1[j - 4], asc, wsc[j]);
      if (RES) cmb[j] = bf16_rne(__int_as_float(j < 4 ? r0[j] : r1[j - 4]) + v[j]);
    }
    if (F32) {
      if (a.out) {
        float* o = reinterpret_cast<float*>(a.out) + i;
        *reinterpret_cast<v4i*>(o) = v4i{__float_as_int(v[0]), __float_as_int(v[1]), __float_as_int(v[2]),
                                         __float_as_int(v[3])};
        *reinterpret_cast<v4i*>(o + 4) = v4i{__float_as_int(v[4]), __float_as_int(v[5]), __float_as_int(v[6]),
                                             __float_as_int(v[7])};
      }
      if (RES) {
        float* o = reinterpret_cast<float*>(a.combined) + i;
        *reinterpret_cast<v4i*>(o) = v4i{__float_as_int(cmb[0]), __float_as_int(cmb[1]), __float_as_int(cmb[2]),
                                         __float_as_int(cmb[3])};
        *reinterpret_cast<v4i*>(o + 4) = v4i{__float_as_int(cmb[4]), __float_as_int(cmb[5]),
                                             __float_as_int(cmb[6]), __float_as_int(cmb[7])};
      }
    } else {
      // BF16 values are the high halves of the BF16-valued floats
      v4i ob, cb;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        ob[j] = (int)((__float_as_uint(v[2 * j]) >> 16) | (__float_as_uint(v[2 * j + 1]) & 0xFFFF0000u));
        cb[j] = (int)((__float_as_uint(cmb[2 * j]) >> 16) | (__float_as_uint(cmb[2 * j + 1]) & 0xFFFF0000u));
      }
      if (a.out) *reinterpret_cast<v4i*>(reinterpret_cast<uint16_t*>(a.out) + i) = ob;
      if (RES) *reinterpret_cast<v4i*>(reinterpret_cast<uint16_t*>(a.combined) + i) = cb;
    }
  }
}

// gemm_dma's tiles and what one costs (ns, fitted to the launches below): fixed +
// K stages x stage with one workgroup on every CU, x pair with two (the tiles
// whose rings take 80 KiB).  A launch runs its tiles in rounds, so the route is
// the tile with the least sum over its rounds: large tiles move the fewest
// operand bytes per product but leave CUs idle in their last round, small
// ones the other way about.  A round that leaves CUs idle runs up to a
// quarter faster (L2 and power are shared).
//
// kDmaTiles, K % 128 == 0: eight waves, and four on 64 x 64.  Measured on MI355X
// with random operands, us per launch (256 x 256 / 256 x 192 / 256 x 128 / 128 x 192 / 128 x 128 / 128 x 64):
// 24576 x 4096 f32 at M = 4096 393 / 417 / 439 / 488 / 537 / -; 6144 x 4096 BF16
// at M = 4096 112 / 97.7 / 103 / 113 / 126 / -, at M = 1024 - / - / 30.3 / 28.1 /
// 38.2 / 39.4, at M = 512 - / - / - / 23.5 / 19.4 / 25.5; 4096 x 4096 f32 with the
// residual at M = 4096 87 / - / 91 / 103 / 112 / -, at M = 1024 - / - / 36 / 29.1
// / 26.9 / 29.8, at M = 512 - / - / 33.7 / 25.7 / 21.0 / 16.7; 4096 x 12288
// likewise at M = 4096 196 / - / 211 / - / 257 / -, at M = 512 - / - / 84 / 72 / 58 /
// 44.7.
//
// With distinct weights, f32 and the residual, 4096 x 4096 on 64 x 64 at M = 129 12.8
// (split K with its slab epilogue 13.6), at M = 256 13.4 (17.4).  Four-wave tiles of
// 128 x 64 and 128 x 32 were within 1 us of those, and slower where they mattered.
// 64 x 128 costs more than 128 x 64 although it moves as much: with distinct
// weights, BF16, 64 x 128 / 128 x 64, 4096 columns at M = 300, K = 4096 15.8 / 14.1
// and K = 8192 28.2 / 24.8, 2560 x 8192 at M = 700 41.2 / 28.2, 3584 x 8192 at M =
// 400 37.6 / 26.6, 6144 x 4096 at M = 129 14.7 / 14.4 and M = 180 16.7 / 14.6, 6144 x
// 5120 at M = 160 21.7 / 17.6.  It leads where 128 x 64 needs twice the rounds
// (10240 x 4096 at M = 129 17.2 / 19.2), and by little at the most tiles of one
// round (8192 x 4096 at M = 129 15.5 / 16.4, M = 180 17.4 / 17.0).
//
// kTailTiles, K % 128 != 0: four waves.  The register-staged kernel that
// these replaced -> the tile the route takes, distinct weights, BF16, M x N x K: 4096 x
// 8000 x 5008 294 -> 163, 2000 x 8000 x 5008 139 -> 87, 1024 x 4096 x 4112 54 -> 30, 512 x
// 6000 x 4112 56 -> 32, 300 x 3000 x 2000 31 -> 10.3, 129 x 4096 x 4112 50 -> 13.2, 77 x
// 5003 x 2000 32 -> 9.0; and gemm_skinny on wider N (skinny_leads): 32 x 12000 x 4112
// 29.6 -> 16.0, 64 x 8192 x 4112 29.0 -> 20.0.
struct DmaTile {
  int bm, bn, wm, wn, sa, sb;
  uint32_t fixed, stage, pair;  // pair 0: one workgroup per CU
};
static const DmaTile kDmaTiles[] = {
    {256, 256, 64, 128, 2, 3, 11000, 1700, 0}, {256, 192, 64, 96, 2, 3, 10000, 1270, 0},
    {256, 128, 64, 64, 2, 4, 7000, 940, 0},    {128, 192, 32, 96, 2, 4, 5000, 740, 0},
    {128, 128, 32, 64, 4, 4, 3000, 590, 0},    {128, 64, 32, 32, 4, 4, 2500, 440, 0},
    {64, 128, 32, 32, 4, 4, 2500, 468, 0},     {64, 64, 32, 32, 4, 4, 3000, 280, 460},
};
static const DmaTile kTailTiles[] = {
    {256, 256, 128, 128, 2, 3, 11000, 1830, 0}, {256, 128, 128, 64, 2, 4, 7000, 1100, 0},
    {128, 128, 64, 64, 2, 3, 5000, 620, 1340},  {128, 64, 64, 32, 3, 4, 4000, 420, 890},
    {64, 64, 32, 32, 4, 4, 3000, 280, 460},
};
static uint64_t launch_ns(const DmaTile& t, uint64_t tiles, uint64_t stages) {
  const uint64_t at_once = t.pair ? 2 * kCus : kCus, rest = tiles % at_once;
  const uint64_t full = t.fixed + stages * (t.pair ? t.pair : t.stage);
  const uint64_t last = rest > kCus ? full : rest ? t.fixed + stages * t.stage * (3 * kCus + rest) / (4 * kCus) : 0;
  return tiles / at_once * full + last;
}

// The cheapest of the tiles for m rows and k, tiles_n(bn) column tiles.
template <size_t N, typename TilesN>
static const DmaTile& cheapest(const DmaTile (&tiles)[N], uint32_t m, uint32_t k, bool residual, TilesN tiles_n) {
  const DmaTile* best = nullptr;
  uint64_t least = ~0ull;
  for (const DmaTile& t : tiles) {
    if (residual && t.wm * t.wn >= 128 * 128) continue;  // !kResidualTile
    const uint64_t c = launch_ns(t, ((uint64_t)m + t.bm - 1) / t.bm * tiles_n(t.bn), ((uint64_t)k + 127) / 128);
    if (c < least) best = &t, least = c;
  }
  return *best;
}

// The route's tile, family and block: the four-wave tiles are kRouteTiled.
static void set_tile(GemmRoute& r, const DmaTile& t) {
  r.bm = t.bm, r.bn = t.bn, r.wm = t.wm, r.wn = t.wn, r.sa = t.sa, r.sb = t.sb;
  r.block = 64 * (t.bm / t.wm) * (t.bn / t.wn);
  r.family = r.block == 256 ? kRouteTiled : kRouteDma;
}

// Whether gemm_dma and gemm_tall take the shape: K in whole 128-byte stages, and
// their 32-bit lane offsets (kMaxK, kMaxCols).
static bool staged_shape(uint32_t n, uint32_t k) { return k % 128 == 0 && k <= kMaxK && n <= kMaxCols; }

// gemm_dma's split-K plan (128 x 128 tiles, two slabs): M > 256 at K >= 8192
// where those tiles, unsplit, would leave more than a third of the CUs idle
// for a long K (4096 x 12288 at M = 512: 36 + 8 us for the slab epilogue
// against 58 unsplit and 44.7 on 128 x 64 tiles).  With more tiles the
// slabs cost more than the CUs they fill: at M = 4096 288 + 64 us against 196
// on 256 x 256 tiles.  A single column of tiles (N <= 128) has the plan at any M for
// calls that ask for it (W8A8_PATH_MFMA with a workspace); AUTO leaves it there
// too (gemm_unsplit_leads).  gemm_tall's plan covers M <= 256.
static bool split_plan(uint32_t m, uint32_t n, uint32_t k, uint32_t& splits) {
  if (m <= 256 || k < 8192 || !staged_shape(n, k) || n % 4 != 0) return false;
  const uint32_t kt = k / 128;
  splits = 2;
  const uint64_t tiles = (uint64_t)((m + 127) / 128) * ((n + 127) / 128);
  return kt % splits == 0 && kt / splits >= 4 && (tiles * 3 <= kCus * 2 || n <= 128);
}

// gemm_narrow's plan: S = 4 waves below K = 8192 and 8 from there (a wave
// walks K / (128 S) stages of 128 bytes), R-deep rings, MB 16-row blocks, LAL
// = ceil(M / 8) activation DMA loads per stage.  It takes M <= 16 on the
// narrow shapes, and M <= 64 where one workgroup per 16 columns fits the
// CUs once at K <= 4096 (4096 x 2048 at M = 40 / 64 5.5 / 6.2 us against gemm_tall
// split K's 7.9 / 7.3, 4096 x 4096 at M = 40 7.8 / 9.3; past 48 rows there see
// split_leads_narrow); the wide shapes (n / 96 >= 224 tiles) keep
// gemm_tall's unsplit 96-column tiles.  Measured on MI355X, graphs of 36
// distinct-weight launches, random operands, against the routes it
// replaced (gemm_tall split-K 4 with its slab epilogue launch, gemm_skinny),
// bit-identical outputs: down 4096 x 12288 at M = 2 / 4 / 8 / 12 / 16
// 10.98 / 11.06 / 11.23 / 11.68 / 12.25 us against 12.64 / 12.72 / 12.77 /
// 13.17 / 13.17 (S = 8); o 4096 x 4096 at M = 2 / 8 / 16 / 24 / 32 5.53 /
// 5.63 / 5.73 / 6.63 / 7.01 against 6.94 / 7.46 / 7.84 / 8.36 / 8.77 (S = 4);
// qkv 6144 x 4096 at M = 2 / 8 / 16 6.98 / 7.48 / 8.09 against 8.30 / 8.98 /
// 9.25 (S = 4; 8.50 / 9.17 / 9.59 with S = 8).  At M = 24 and 32 down and
// qkv are level or slower than gemm_tall (down 13.78 / 15.12 against 13.59 /
// 14.03) and keep it.  gate_up (24576 x 4096, 1,536 workgroups) measured
// slower on it (M = 4 / 8 / 16 19.31 / 19.86 / 21.74 us against 18.23 /
// 18.01 / 17.41 on the 96-column tiles).  Deeper rings (5) and 16 waves
// measured level or slower.  These down figures are for contiguous K slices;
// the interleaved order the kernel now takes at S = 8 runs 2-3% faster.
static bool narrow_plan(uint32_t m, uint32_t n, uint32_t k, int& S, int& R, int& MB, int& LAL) {
  if (m == 0 || m > 64 || (n + 95) / 96 >= 224) return false;
  S = k >= 8192 ? 8 : 4;
  if (k % (128u * S) != 0) return false;
  if (m > 16 && !(k <= 4096 && (n + 15) / 16 <= 256)) return false;
  MB = (int)((m + 15) / 16);  // more than one only at S = 4 (K <= 4096)
  LAL = (int)((m + 7) / 8);
  R = MB <= 3 ? 4 : 3;  // LDS
  return true;
}

static bool tall_plan(uint32_t m, uint32_t n, uint32_t k, int& bn, uint32_t& splits, int& ma);

// Whether, with a workspace, gemm_tall's split K beats gemm_narrow on a shape of
// narrow_plan: four 16-row blocks at the longest K, whose rings are three deep, and
// which pull 64 activation rows over all of K into every CU.  Measured on MI355X
// with distinct weights, gemm_narrow / split us, 4096 columns x K = 4096, BF16 and f32
// with the residual: M = 48 8.3 / 8.6 and 9.2 / 9.2, M = 52 level and 9.8 / 9.1, M = 64
// 9.0 / 8.7 and 10.3 / 9.3; 512 columns M = 56 7.9 / 7.4, 1024 M = 56 7.9 / 7.6, M = 64 8.2 / 7.9; not 2048
// columns at M = 57 8.2 / 8.4, 3000 at M = 64 8.7 / 9.2 (split K's 64-column tiles fill the CUs
// less well there); at K = 3584 level or slower.
static bool split_leads_narrow(uint32_t m, uint32_t n, uint32_t k) {
  int bn, ma;
  uint32_t splits;
  if (n > 1536 && n <= 3050) return false;
  return m > (n > 3900 ? 48u : n > 3500 || n <= 1024 ? 52u : 56u) && k > 3584 && tall_plan(m, n, k, bn, splits, ma) && splits > 1;
}

// gemm_tall plan for 1 <= m <= 256 (measured on MI355X on the Qwen3-8B
// projection shapes at M = 16, 64, 65, 80, 100, 128 and 129): 96-column
// tiles when they alone give about one tile per CU; otherwise split K four
// ways (two when K is short), with 96- or 64-column tiles, to reach about one
// workgroup per CU.  For 64 < m <= 128 one 160-row tile streams the weights
// once where gemm_dma's two 64-row tiles stream them twice (gate_up at
// M = 100 24.6-24.9 against 33.3-34.1 us, down 20.7 against 23.3-23.5), and
// with streamed slabs the split route also beats gemm_dma's split-K 2 on
// qkv and o (qkv at M = 65 / 100 / 128 12.6 / 14.1 / 14.5 against
// 13.2-13.3 / 14.6 / 15.5, o 10.9 / 11.6 / 12.7 against 12.0 / 12.7 / 13.2).
// At small m the plan applies to the wide shapes and to long K at any m,
// where it beats gemm_skinny (graphs of 16 distinct-weight launches, random
// operands, m = 1..6: gate_up 17.9-18.1 against 21.2-24.0 us, down at
// K = 12288 13.1-13.5 against 16.7-17.1).  At K = 4096 on narrow N the
// skinny kernel (one workgroup per 16 columns) led while its grid fits the
// CUs once: o (4096 columns) at m = 2 / 4 / 8 / 12 / 16 / 24 7.1 / 7.2 /
// 7.4 / 7.6 / 7.9 / 9.6 us against 7.8 / 7.8 / 8.0 / 8.0 / 8.2 / 9.0; qkv
// (6144 columns) 8.4 / 8.8 / 9.6 / 10.5 / 11.5 against 8.6 / 8.8 / 9.0 /
// 9.1 / 9.3, so it takes this plan from m = 8, o from m = 24.  gemm_narrow's
// plan, checked first, now takes the small batches on narrow N.
// Returns false when no plan applies (the gemm_dma or gemm_skinny routes
// then run).  ma: the M tile (64, 160 or 256 rows).
static bool tall_plan(uint32_t m, uint32_t n, uint32_t k, int& bn, uint32_t& splits, int& ma) {
  if (m == 0 || m > 256 || !staged_shape(n, k)) return false;
  ma = m <= 64 ? 64 : m <= 160 ? 160 : 256;
  const uint32_t kt = k / 128, t96 = (n + 95) / 96;
  if (t96 >= 224) {
    bn = 96;
    splits = 1;
    return true;
  }
  if (n % 4 != 0) return false;  // the split-K epilogue works on column quads
  if (k < 8192 && (m < 8 || (m < 24 && (n + 15) / 16 <= 256))) return false;
  splits = (kt % 4 == 0 && kt / 4 >= 4) ? 4 : (kt % 2 == 0 && kt / 2 >= 4) ? 2 : 1;
  if (splits == 1) return false;
  bn = t96 * splits >= 224 ? 96 : 64;
  return true;
}

// Whether one unsplit launch of gemm_dma's small tiles runs a shape of gemm_tall's
// split plan faster than the split GEMM and its slab epilogue: above 64 rows, up
// to a K that grows with the rows and with the slabs.  Always where the split
// grid takes a second round, and later where only two slabs divide K.
// Measured on MI355X with distinct weights, BF16, split / unsplit us at K = 2048 /
// 3072 / 4096 / 5120 / 8192:
//   1024 cols, M = 65    7.2 /  7.6    8.0 /  9.7    8.9 / 11.7    9.9 / 13.8   12.2 / 19.9
//              M = 129   8.3 /  7.6    9.5 /  9.6   10.3 / 11.7   11.5 / 13.8   14.2 / 19.9
//              M = 256   9.4 /  7.7   10.7 /  9.9   11.4 / 11.9   13.5 / 15.0   16.2 / 20.5
//   4096 cols, M = 65    7.9 /  7.8    8.8 /  9.9    9.6 / 12.0   10.7 / 14.4   13.1 / 20.7
//              M = 100   8.6 /  7.8    9.7 / 10.1   10.4 / 12.2   12.5 / 15.3   14.2 / 21.1
//              M = 129  10.0 /  7.8   11.2 /  9.9   12.1 / 12.0   13.4 / 14.4   16.4 / 20.7
//              M = 193  10.9 /  7.8   12.6 / 10.0   13.7 / 12.1   15.4 / 14.6   18.9 / 21.2
//              M = 256  13.2 /  8.0   14.7 / 10.4   16.2 / 12.5   17.9 / 16.1   22.2 / 21.8
//   6144 cols, M = 129  11.3 /  9.3   13.4 / 12.4   14.6 / 14.5   16.3 / 17.3   20.6 / 25.2
//              M = 256  17.2 / 10.1   19.6 / 13.9   21.5 / 16.2   23.1 / 22.4   28.6 / 29.9
//   8192 cols, M = 129  17.6 /  9.6   20.9 / 12.7   23.2 / 15.5   26.3 / 20.1   33.3 / 26.6
// Two slabs, unsplit over split at K = 4352 / 5376 / 7936: M = 65 0.95-0.99 / 0.99-1.02 /
// 1.04-1.06, M = 129 0.83-0.87 / 0.84-0.89 / 0.90-0.92 (1024 to 4096 columns).
// Above 256 rows: split_plan's single column of tiles past its share of the CUs (64
// columns, M = 22,000 / 33,000, K = 8192 48 / 83 split, 27 / 57 unsplit; within it the pair is
// level at K = 8192 and leads beyond, M = 300 to 1,500 at K = 16384 31 / 35).
bool gemm_unsplit_leads(uint32_t m, uint32_t n, uint32_t k) {
  int bn, ma;
  uint32_t splits;
  if (m > 256) return split_plan(m, n, k, splits) && (uint64_t)((m + 127) / 128) * 3 > kCus * 2 && n <= 128;
  if (m <= 64 || k > 8192 || !tall_plan(m, n, k, bn, splits, ma) || splits == 1) return false;
  if ((n + bn - 1) / bn * splits > kCus) return true;
  if (splits == 2) return m > 100 || k <= 5376;
  return 2000 * k <= 27000 * m + 9 * m * std::min(n, 4096u);
}

size_t gemm_workspace_bytes(uint32_t m, uint32_t n, uint32_t k) {
  int tile;
  uint32_t splits;
  int ma;
  {
    int S, R, MB, LAL;
    if (narrow_plan(m, n, k, S, R, MB, LAL) && !split_leads_narrow(m, n, k)) return 0;
  }
  if (tall_plan(m, n, k, tile, splits, ma)) return splits > 1 ? (size_t)splits * m * n * sizeof(int32_t) : 0;
  if (!split_plan(m, n, k, splits)) return 0;
  return (size_t)splits * m * n * sizeof(int32_t);
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// gemm_tall's split-K slab sets of at least this many bytes are streamed:
// written with non-temporal stores (EP_SLAB) and read back non-temporally.
// Measured on MI355X (graphs of 16 distinct-weight launches, GEMM + slab
// epilogue, plain -> streamed): qkv at M = 255 23.6 -> 19.7-20.2 us, o at
// M = 255 19.1 -> 15.9, down at M = 200 26.3 -> 25.1, qkv at M = 129
// 19.4 -> 16.0, o at M = 129 14.4 -> 13.8-14.1, qkv at M = 40 13.6 -> 12.9.
// The streamed GEMM itself runs 1.2-1.3 us faster (no dirty slab lines left
// in L2 at its end).  Smaller sets, whose epilogue is latency-bound, lose
// (down at M = 32, 2 MiB: 16.6 -> 17.0; at M = 16, 1 MiB: 15.4 -> 15.9), and
// so does gemm_dma's split route (down at M = 512 38.3 -> 41.0, at M = 300
// 32.0 -> 33.2): both keep the default policy.
constexpr size_t kSlabStreamBytes = size_t(3) << 20;

static bool stream_slabs(const GemmArgs& a, uint32_t splits) {
  return (size_t)splits * a.m * a.n * sizeof(int32_t) >= kSlabStreamBytes;
}

template <int EP, bool NT>
static void launch_epilogue(hipStream_t st, const GemmArgs& a, uint32_t splits, bool wide) {
  const uint32_t rows = std::min<uint32_t>(a.m, 65535);
  if (wide)
    hipLaunchKernelGGL((splitk_epilogue8<EP, NT>), dim3((a.n / 8 + 255) / 256, rows), dim3(256), 0, st, a,
                       a.partials, splits);
  else
    hipLaunchKernelGGL((splitk_epilogue<EP, NT>), dim3((a.n / 4 + 255) / 256, rows), dim3(256), 0, st, a,
                       a.partials, splits);
}

// 8 columns per split-K epilogue thread above M = 200 when every row of
// every operand starts 16-byte aligned (n % 8 == 0 and aligned bases); 4
// otherwise.  The epilogue is latency-bound: up to M = 200 twice the threads
// with half the loads each finish sooner.  Measured on MI355X, graphs of 16
// distinct-weight launches, GEMM + epilogue, 8 -> 4 columns: M = 64 o
// 10.3 -> 9.7 us, M = 100 qkv 14.4 -> 13.5, M = 129 qkv 15.6-15.8 -> 14.9,
// o 13.5-13.9 -> 13.1, down 22.6-24.1 -> 22.0, M = 200 qkv 18.7 -> 17.7;
// but M = 255 o 15.9-16.1 -> 17.1, and level on gemm_dma's split route at
// M = 300 and 512.  Two columns per thread (256- or 512-thread workgroups)
// and four with 1,024-thread workgroups measured level or slower from M = 24
// to 200 (M = 129 o 12.28-12.44 against 12.24 us, down 21.6-21.8 against
// 21.5).
static bool wide_epilogue(const GemmArgs& a) {
  return a.m > 200 && a.n % 8 == 0 && aligned16(a.partials) && aligned16(a.out) &&
         (a.out_dtype == W8A8_OUT_I32 || aligned16(a.ws)) &&
         (!a.residual || (aligned16(a.residual) && aligned16(a.combined)));
}

template <bool NT>
static hipError_t launch_splitk_epilogue(hipStream_t st, const GemmArgs& a, uint32_t splits) {
  if (splits < 1 || splits > kMaxSplits) return hipErrorInvalidValue;
  const bool wide = wide_epilogue(a);
  if (a.out_dtype == W8A8_OUT_I32)
    launch_epilogue<EP_I32, NT>(st, a, splits, wide);
  else if (a.out_dtype == W8A8_OUT_F32 && a.residual)
    launch_epilogue<EP_F32_RES, NT>(st, a, splits, wide);
  else if (a.out_dtype == W8A8_OUT_F32)
    launch_epilogue<EP_F32, NT>(st, a, splits, wide);
  else if (a.residual)
    launch_epilogue<EP_BF16_RES, NT>(st, a, splits, wide);
  else
    launch_epilogue<EP_BF16, NT>(st, a, splits, wide);
  return hipGetLastError();
}

// Split-K launch: `gemm` launches the split GEMM into a.partials, given the
// slab mode as a compile-time constant; the slab epilogue follows.  Both
// take the same slab policy (nt: streamed).
template <typename Launch>
static hipError_t launch_slabs(hipStream_t st, const GemmArgs& a, uint32_t splits, bool nt, Launch gemm) {
  GemmArgs p = a;
  p.out = a.partials;
  p.out_dtype = W8A8_OUT_I32;
  if (nt) gemm(std::integral_constant<int, EP_SLAB>{}, p);
  else gemm(std::integral_constant<int, EP_I32>{}, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return nt ? launch_splitk_epilogue<true>(st, a, splits) : launch_splitk_epilogue<false>(st, a, splits);
}

template <int BM, int BN, int WM, int WN, int SA, int SB>
static hipError_t launch_split(hipStream_t st, const GemmArgs& a, uint32_t splits) {
  const uint32_t tm = (a.m + BM - 1) / BM, tn = (a.n + BN - 1) / BN;
  return launch_slabs(st, a, splits, false, [&](auto ep, const GemmArgs& p) {
    hipLaunchKernelGGL((gemm_dma<BM, BN, WM, WN, SA, SB, decltype(ep)::value>), dim3(tm * tn * splits),
                       dim3(512), 0, st, p, tm, tn, splits, NoGroup{});
  });
}

template <int BN, int SA, int SB, int MA>
static hipError_t launch_tall(hipStream_t st, const GemmArgs& a, uint32_t splits) {
  const uint32_t tn = (a.n + BN - 1) / BN;
  const dim3 grid(tn * splits), block(512);
  if (splits > 1)
    return launch_slabs(st, a, splits, stream_slabs(a, splits), [&](auto ep, const GemmArgs& p) {
      hipLaunchKernelGGL((gemm_tall<BN, SA, SB, MA, decltype(ep)::value, false>), grid, block, 0, st, p, tn, splits,
                         nullptr, NoGroup{});
    });
  if (a.out_dtype == W8A8_OUT_I32)
    hipLaunchKernelGGL((gemm_tall<BN, SA, SB, MA, EP_I32, kRotateK>), grid, block, 0, st, a, tn, 1u, nullptr, NoGroup{});
  else if (a.out_dtype == W8A8_OUT_F32 && a.residual)
    hipLaunchKernelGGL((gemm_tall<BN, SA, SB, MA, EP_F32_RES, kRotateK>), grid, block, 0, st, a, tn, 1u, nullptr, NoGroup{});
  else if (a.out_dtype == W8A8_OUT_F32)
    hipLaunchKernelGGL((gemm_tall<BN, SA, SB, MA, EP_F32, kRotateK>), grid, block, 0, st, a, tn, 1u, nullptr, NoGroup{});
  else if (a.residual)
    hipLaunchKernelGGL((gemm_tall<BN, SA, SB, MA, EP_BF16_RES, kRotateK>), grid, block, 0, st, a, tn, 1u, nullptr, NoGroup{});
  else
    hipLaunchKernelGGL((gemm_tall<BN, SA, SB, MA, EP_BF16, kRotateK>), grid, block, 0, st, a, tn, 1u, nullptr, NoGroup{});
  return hipGetLastError();
}

// Diagnostics: gemm_tall with the per-wave clock stamps (TIMED), BF16
// outputs without a residual; the split-K epilogue follows as in launch_tall.
template <int BN, int SA, int SB, int MA>
static hipError_t launch_tall_timed(hipStream_t st, const GemmArgs& a, uint32_t splits, uint64_t* stamps) {
  const uint32_t tn = (a.n + BN - 1) / BN;
  const dim3 grid(tn * splits), block(512);
  if (splits > 1)
    return launch_slabs(st, a, splits, stream_slabs(a, splits), [&](auto ep, const GemmArgs& p) {
      hipLaunchKernelGGL((gemm_tall<BN, SA, SB, MA, decltype(ep)::value, false, true>), grid, block, 0, st, p, tn,
                         splits, stamps, NoGroup{});
    });
  hipLaunchKernelGGL((gemm_tall<BN, SA, SB, MA, EP_BF16, kRotateK, true>), grid, block, 0, st, a, tn, 1u, stamps, NoGroup{});
  return hipGetLastError();
}

// ---------------------------------------------------------------- dispatch
// The route of one GEMM call (see GemmRoute).
// Where no plan runs, whether gemm_skinny's K split over a workgroup's waves beats
// gemm_dma's small tiles, which walk K in one piece: always up to 16 rows; with up to
// one 16-column workgroup per CU to 32 rows, and to 64 with a K tail (whose rows
// cross cache lines, which costs the DMA more) or a short K; with twice the
// columns at the shortest K.  Measured on MI355X with distinct weights, BF16, M x N x
// K, gemm_skinny / gemm_dma us: 17 x 1024 x 8208 16.4 / 21.3, 32 x 512 x 16016 37 / 44,
// 32 x 4096 x 8192 15.8 / 20.6, 33 x 4096 x 2064 8.5 / 8.8, 48 x 1024 x 4112 13.4 / 16.1,
// 64 x 1024 x 12304 41 / 50, 64 x 4096 x 16016 57 / 66, 48 x 4096 x 384 3.8 / 5.1, 64 x 4096 x
// 384 4.2 / 5.0, 24 x 6144 x 1040 6.2 / 6.2, 32 x 8192 x 528 4.5 / 4.9, 48 x 6144 x 384 4.6 /
// 5.2; not taken: 33 x 1024 x 8192 23.3 / 19.8, 64 x 4096 x 16384 43.8 / 39.0, 48 x 4096 x
// 1152 6.5 / 6.1, 64 x 4096 x 640 5.4 / 5.0, 32 x 6144 x 8192 28 / 21, 32 x 6144 x 1040 6.9 / 6.3.
static bool skinny_leads(uint32_t m, uint32_t n, uint32_t k) {
  if (m <= 16) return true;
  if (m > 64 || n > 32 * kCus) return false;
  if (n <= 16 * kCus) return m <= 32 || k % 128 != 0 || k <= (m <= 48 ? 896u : 384u);
  return k <= (m <= 24 ? 1040u : m <= 32 ? 640u : m <= 48 ? 384u : 0u);
}

GemmRoute gemm_route(const GemmArgs& a) {
  GemmRoute r{};
  r.splits = 1;
  r.epi_cols = 4;
  r.grid_y = 1;
  r.block = 512;
  if (a.m == 0 || a.n == 0) return r;
  {
    int S, R, MB, LAL;
    const size_t slabs = 4 * (size_t)a.m * a.n * sizeof(int32_t);
    const bool split = a.partials && a.partial_bytes >= slabs && split_leads_narrow(a.m, a.n, a.k);
    if (!split && narrow_plan(a.m, a.n, a.k, S, R, MB, LAL)) {
      r.family = kRouteNarrow;
      r.mt = MB;
      r.s = S;
      r.u = LAL;
      r.sa = R;
      r.grid_x = (a.n + 15) / 16;
      r.block = 64 * S;
      return r;
    }
  }
  // m <= 256 goes to gemm_tall when its plan applies.
  // Otherwise, for small m: from m = 8 the 8-wave kernel with 64-row tiles
  // streams the weights faster when n gives at least 128 tiles; below that
  // the skinny kernel's split-K keeps more CUs busy.
  const bool wide = a.m >= 8 && staged_shape(a.n, a.k) && (a.n + 127) / 128 >= 128;
  {
    int tile, ma;
    uint32_t splits;
    if (tall_plan(a.m, a.n, a.k, tile, splits, ma) &&
        (splits == 1 || (a.partials && a.partial_bytes >= (size_t)splits * a.m * a.n * sizeof(int32_t)))) {
      // Ring depths four and four for the 64- and 160-row tiles.  Measured on
      // MI355X, graphs of 16 distinct-weight launches (split routes: GEMM +
      // epilogue), from 8 / 8 and 4 / 8 (64 rows) and 5 / 5 and 4 / 6 (160
      // rows): M = 16 qkv 10.25 -> 9.3 us, o 8.56 -> 8.24, down 13.7 -> 13.2,
      // gate_up 18.1 -> 17.3; M = 64 qkv 11.6-11.8 -> 10.4, o 9.6-9.8 -> 8.8,
      // down 15.4-16.0 -> 14.9, gate_up 19.7-20.0 -> 19.0-19.2; M = 80 down
      // 18.7-19.5 -> 16.9; M = 100 qkv 13.2 -> 12.4-12.6, o 11.2 -> 10.4,
      // down 19.6-19.8 -> 17.7-18.1; M = 129 qkv 14.7-14.8 -> 14.0-14.3, o
      // 13.1-13.2 -> 12.4-12.6, gate_up 28.7-28.9 -> 27.0-28.1; M = 160 down
      // level.  6 / 6, 5 / 5, 4 / 5, 3 / 4 and 3 / 3 measured in between.  The
      // 256-row tile: 2 / 4 for the unsplit 96-column tiles (gate_up at
      // M = 200 33.7-35.1 -> 31.5-32.9 us, M = 255 37.6-37.9 -> 36.1-37.1
      // from 3 / 3), 3 / 3 and 4 / 4 for the split routes (2 / 3, 2 / 4 and
      // 3 / 4 level or slower there).
      r.family = kRouteTall;
      r.bn = tile;
      r.ma = ma;
      r.splits = splits;
      r.sa = r.sb = 4;
      if (ma == 256 && tile == 96) {
        r.sa = splits > 1 ? 3 : 2;
        r.sb = splits > 1 ? 3 : 4;
      }
      r.grid_x = (a.n + tile - 1) / tile * splits;
      if (splits > 1) {
        r.nt_slabs = stream_slabs(a, splits);
        r.epi_cols = wide_epilogue(a) ? 8 : 4;
      }
      return r;
    }
  }
  if (!wide && skinny_leads(a.m, a.n, a.k)) {
    r.family = kRouteSkinny;
    r.mt = a.m <= 16 ? 1 : a.m <= 32 ? 2 : 4;
    r.s = 4;
    r.u = a.m <= 32 ? 4 : 2;
    r.grid_x = (a.n + 15) / 16;
    r.block = 64 * r.s;
    return r;
  }
  auto tiles_n = [&](uint32_t bn) { return ((uint64_t)a.n + bn - 1) / bn; };
  const bool residual = a.residual != nullptr;
  uint32_t splits;
  if (!staged_shape(a.n, a.k)) {
    set_tile(r, cheapest(kTailTiles, a.m, a.k, residual, tiles_n));
  } else if (a.partials && split_plan(a.m, a.n, a.k, splits) &&
             a.partial_bytes >= (size_t)splits * a.m * a.n * sizeof(int32_t)) {
    set_tile(r, kDmaTiles[4]);
    r.splits = splits;
    r.epi_cols = wide_epilogue(a) ? 8 : 4;
  } else {
    set_tile(r, cheapest(kDmaTiles, a.m, a.k, residual, tiles_n));
  }
  r.grid_x = (a.m + r.bm - 1) / r.bm * ((a.n + r.bn - 1) / r.bn) * r.splits;
  return r;
}

size_t gemm_timeline_waves(const GemmArgs& a) {
  const GemmRoute r = gemm_route(a);
  return r.family == kRouteTall ? (size_t)r.grid_x * 8 : 0;
}

hipError_t launch_gemm_timeline(hipStream_t st, const GemmArgs& a, uint64_t* stamps) {
  const GemmRoute r = gemm_route(a);
  if (r.family != kRouteTall || a.out_dtype != W8A8_OUT_BF16 || a.residual) return hipErrorInvalidValue;
  if (r.ma == 64)
    return r.bn == 96 ? launch_tall_timed<96, 4, 4, 64>(st, a, r.splits, stamps)
                      : launch_tall_timed<64, 4, 4, 64>(st, a, r.splits, stamps);
  if (r.ma == 160)
    return r.bn == 96 ? launch_tall_timed<96, 4, 4, 160>(st, a, r.splits, stamps)
                      : launch_tall_timed<64, 4, 4, 160>(st, a, r.splits, stamps);
  if (r.bn == 96)
    return r.splits > 1 ? launch_tall_timed<96, 3, 3, 256>(st, a, r.splits, stamps)
                        : launch_tall_timed<96, 2, 4, 256>(st, a, r.splits, stamps);
  return launch_tall_timed<64, 4, 4, 256>(st, a, r.splits, stamps);
}

template <int MB, int LAL, int S, int R, int NB = 1, class G>
static hipError_t launch_narrow_as(hipStream_t st, const GemmArgs& a, const G& g, uint32_t grid) {
  constexpr bool GROUP = std::is_same_v<G, GemmGroup>;
  hipLaunchKernelGGL((gemm_narrow<MB, LAL, S, R, GROUP, NB>), dim3(grid), dim3(64 * S), 0, st, a, g);
  return hipGetLastError();
}

// The instantiations the plans can ask for: S = 4 with one to four 16-row
// blocks, S = 8 (K >= 8192) with one; LAL = ceil(M / 8); NB = 2 from two blocks
// on, for groups.
template <int NB, class G>
static hipError_t launch_narrow(hipStream_t st, const GemmArgs& a, const G& g, const GemmRoute& r) {
  const uint32_t n = r.grid_x;
  if (r.s == 4) {
    switch (r.u) {
      case 3: return launch_narrow_as<2, 3, 4, 4, NB>(st, a, g, n);
      case 4: return launch_narrow_as<2, 4, 4, 4, NB>(st, a, g, n);
      case 5: return launch_narrow_as<3, 5, 4, 4, NB>(st, a, g, n);
      case 6: return launch_narrow_as<3, 6, 4, 4, NB>(st, a, g, n);
      case 7: return launch_narrow_as<4, 7, 4, 3, NB>(st, a, g, n);
      case 8: return launch_narrow_as<4, 8, 4, 3, NB>(st, a, g, n);
    }
    if constexpr (NB == 1)
      return r.u == 1 ? launch_narrow_as<1, 1, 4, 4>(st, a, g, n) : launch_narrow_as<1, 2, 4, 4>(st, a, g, n);
  } else if constexpr (NB == 1) {
    return r.u == 1 ? launch_narrow_as<1, 1, 8, 4>(st, a, g, n) : launch_narrow_as<1, 2, 8, 4>(st, a, g, n);
  }
  return hipErrorInvalidValue;
}

static hipError_t launch_tail(hipStream_t st, const GemmArgs& a, const GemmRoute& r) {
  if (r.bm == 256 && r.bn == 256) return launch_dma<256, 256, 128, 128, 2, 3, 4, true>(st, a);
  if (r.bm == 256) return launch_dma<256, 128, 128, 64, 2, 4, 4, true>(st, a);
  if (r.bm == 128 && r.bn == 128) return launch_dma<128, 128, 64, 64, 2, 3, 4, true>(st, a);
  if (r.bm == 128) return launch_dma<128, 64, 64, 32, 3, 4, 4, true>(st, a);
  return launch_dma<64, 64, 32, 32, 4, 4, 4, true>(st, a);
}

hipError_t launch_gemm(hipStream_t st, const GemmArgs& a) {
  const GemmRoute r = gemm_route(a);
  auto is = [&](int bm, int bn, int wm, int wn, int sa, int sb) {
    return r.bm == bm && r.bn == bn && r.wm == wm && r.wn == wn && r.sa == sa && r.sb == sb;
  };
  switch (r.family) {
    case kRouteNone:
      return hipSuccess;
    case kRouteTall:
      if (r.ma == 64)
        return r.bn == 96 ? launch_tall<96, 4, 4, 64>(st, a, r.splits) : launch_tall<64, 4, 4, 64>(st, a, r.splits);
      if (r.ma == 160)
        return r.bn == 96 ? launch_tall<96, 4, 4, 160>(st, a, r.splits) : launch_tall<64, 4, 4, 160>(st, a, r.splits);
      if (r.bn == 96)
        return r.splits > 1 ? launch_tall<96, 3, 3, 256>(st, a, r.splits) : launch_tall<96, 2, 4, 256>(st, a, r.splits);
      return launch_tall<64, 4, 4, 256>(st, a, r.splits);
    case kRouteNarrow:
      return launch_narrow<1>(st, a, NoGroup{}, r);
    case kRouteSkinny:
      if (r.mt == 1) hipLaunchKernelGGL((gemm_skinny<1, 4, 4>), dim3(r.grid_x, 1), dim3(r.block), 0, st, a);
      else if (r.mt == 2) hipLaunchKernelGGL((gemm_skinny<2, 4, 4>), dim3(r.grid_x, 1), dim3(r.block), 0, st, a);
      else hipLaunchKernelGGL((gemm_skinny<4, 4, 2>), dim3(r.grid_x, 1), dim3(r.block), 0, st, a);
      return hipGetLastError();
    case kRouteDma:
      if (r.splits > 1) return launch_split<128, 128, 32, 64, 4, 4>(st, a, r.splits);
      if (is(256, 256, 64, 128, 2, 3)) return launch_dma<256, 256, 64, 128, 2, 3>(st, a);
      if (is(256, 192, 64, 96, 2, 3)) return launch_dma<256, 192, 64, 96, 2, 3>(st, a);
      if (is(256, 128, 64, 64, 2, 4)) return launch_dma<256, 128, 64, 64, 2, 4>(st, a);
      if (is(128, 192, 32, 96, 2, 4)) return launch_dma<128, 192, 32, 96, 2, 4>(st, a);
      if (is(128, 128, 32, 64, 4, 4)) return launch_dma<128, 128, 32, 64, 4, 4>(st, a);
      if (is(128, 64, 32, 32, 4, 4)) return launch_dma<128, 64, 32, 32, 4, 4>(st, a);
      return launch_dma<64, 128, 32, 32, 4, 4>(st, a);
    case kRouteTiled:
      return staged_shape(a.n, a.k) ? launch_dma<64, 64, 32, 32, 4, 4, 4>(st, a) : launch_tail(st, a, r);
  }
  return hipErrorInvalidValue;
}

// ---------------------------------------------------------------- grouped
template <int BN, int SA, int SB, int MA>
static hipError_t launch_tall_group(hipStream_t st, const GemmArgs& a, const GemmGroup& g, uint32_t tn) {
  auto k = a.out_dtype == W8A8_OUT_I32   ? gemm_tall<BN, SA, SB, MA, EP_I32, kRotateK, false, true>
           : a.out_dtype == W8A8_OUT_F32 ? gemm_tall<BN, SA, SB, MA, EP_F32, kRotateK, false, true>
                                         : gemm_tall<BN, SA, SB, MA, EP_BF16, kRotateK, false, true>;
  hipLaunchKernelGGL(k, dim3(tn), dim3(512), 0, st, a, tn, 1u, nullptr, g);
  return hipGetLastError();
}

template <int BM, int BN, int WM, int WN, int SA, int SB, int NW = 8>
static hipError_t launch_dma_group(hipStream_t st, const GemmArgs& a, const GemmGroup& g, uint32_t tn) {
  const uint32_t tm = (a.m + BM - 1) / BM;
  auto k = a.out_dtype == W8A8_OUT_I32   ? gemm_dma<BM, BN, WM, WN, SA, SB, EP_I32, true, NW>
           : a.out_dtype == W8A8_OUT_F32 ? gemm_dma<BM, BN, WM, WN, SA, SB, EP_F32, true, NW>
                                         : gemm_dma<BM, BN, WM, WN, SA, SB, EP_BF16, true, NW>;
  hipLaunchKernelGGL(k, dim3(tm * tn), dim3(64 * NW), 0, st, a, tm, tn, 1u, g);
  return hipGetLastError();
}

// The grouped route: the single projection's unsplit routes on the siblings'
// columns together (groups have no workspace), so a group fills the chip where
// its matrices alone would not, and pays one launch.  Measured on MI355X with
// distinct weights, BF16, one launch per matrix (dot4 up to M = 4) -> this, us: gate
// and up (12288 x 4096 each) at M = 4 20.8 -> 17.4, M = 32 46.4 -> 17.4, M = 129 57.3 ->
// 28.0, M = 512 66.0 -> 52.1, M = 4096 435 -> 367; q, k and v (4096 + 1024 + 1024) at M = 4 8.8
// -> 7.5, M = 32 19.3 -> 9.6, M = 129 44.8 -> 14.9, M = 512 47.6 -> 22.4, M = 4096 173 -> 104.
GemmRoute gemm_group_route(uint32_t m, uint32_t k, const uint32_t* n, int count) {
  GemmRoute r{};
  r.splits = 1;
  r.grid_y = 1;
  r.block = 512;
  uint64_t total = 0;
  for (int i = 0; i < count; ++i) total += n[i];
  if (total > kMaxCols || !staged_shape((uint32_t)total, k)) return r;
  auto tiles = [&](uint32_t bn) {
    uint64_t t = 0;
    for (int i = 0; i < count; ++i) t += (n[i] + bn - 1) / bn;
    return t;
  };
  int S, R, MB, LAL;
  if (narrow_plan(m, (uint32_t)total, k, S, R, MB, LAL)) {
    r.family = kRouteNarrow;
    r.mt = MB, r.s = S, r.u = LAL, r.sa = R;
    r.bn = 16;
    r.block = 64 * S;
    r.grid_x = (uint32_t)tiles(16);
    return r;
  }
  // Two 16-column blocks per workgroup where that fits the CUs once: 6144 x 4096
  // at M = 24 / 32 / 48 / 64 7.9 / 8.1 / 9.6 / 10.5 us against 11.6 / 11.2 / 11.5 /
  // 11.5 on 64 x 64 tiles.
  if (m > 16 && m <= 64 && k <= 4096 && k % 512 == 0 && tiles(32) <= kCus) {
    r.family = kRouteNarrow;
    r.mt = (int)((m + 15) / 16), r.s = 4, r.u = (int)((m + 7) / 8), r.sa = m <= 48 ? 4 : 3;
    r.bn = 32;
    r.block = 256;
    r.grid_x = (uint32_t)tiles(32);
    return r;
  }
  if (m <= 256 && tiles(96) >= 224) {
    r.family = kRouteTall;
    r.ma = m <= 64 ? 64 : m <= 160 ? 160 : 256;
    r.bn = 96;
    r.sa = r.ma == 256 ? 2 : 4, r.sb = 4;
    r.grid_x = (uint32_t)tiles(r.bn);
    return r;
  }
  set_tile(r, cheapest(kDmaTiles, m, k, false, tiles));
  const uint64_t grid = (m + r.bm - 1) / r.bm * tiles(r.bn);
  if (grid > 0x7fffffu) return GemmRoute{};
  r.grid_x = (uint32_t)grid;
  return r;
}

hipError_t launch_gemm_group(hipStream_t st, const GemmArgs& a, GemmGroup& g) {
  const GemmRoute r = gemm_group_route(a.m, a.k, g.n, g.count);
  if (r.family == kRouteNone) return hipErrorInvalidValue;
  uint32_t tn = 0;
  for (int i = 0; i <= kMaxGroup; ++i) {
    g.tbegin[i] = tn;
    if (i < g.count) tn += (g.n[i] + r.bn - 1) / r.bn;
  }
  if (r.family == kRouteNarrow) return r.bn == 32 ? launch_narrow<2>(st, a, g, r) : launch_narrow<1>(st, a, g, r);
  if (r.family == kRouteTall) {
    return r.ma == 64    ? launch_tall_group<96, 4, 4, 64>(st, a, g, tn)
           : r.ma == 160 ? launch_tall_group<96, 4, 4, 160>(st, a, g, tn)
                         : launch_tall_group<96, 2, 4, 256>(st, a, g, tn);
  }
  if (r.family == kRouteTiled) return launch_dma_group<64, 64, 32, 32, 4, 4, 4>(st, a, g, tn);
  if (r.bm == 256 && r.bn == 256) return launch_dma_group<256, 256, 64, 128, 2, 3>(st, a, g, tn);
  if (r.bm == 256 && r.bn == 192) return launch_dma_group<256, 192, 64, 96, 2, 3>(st, a, g, tn);
  if (r.bm == 256) return launch_dma_group<256, 128, 64, 64, 2, 4>(st, a, g, tn);
  if (r.bm == 64) return launch_dma_group<64, 128, 32, 32, 4, 4>(st, a, g, tn);
  if (r.bn == 192) return launch_dma_group<128, 192, 32, 96, 2, 4>(st, a, g, tn);
  if (r.bn == 128) return launch_dma_group<128, 128, 32, 64, 4, 4>(st, a, g, tn);
  return launch_dma_group<128, 64, 32, 32, 4, 4>(st, a, g, tn);
}

}  // namespace w8a8
