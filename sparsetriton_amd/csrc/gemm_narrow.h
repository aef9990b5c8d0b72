// Gather-GEMM over a tile plan for layers with few channels (forward and
// input gradient): all K weight slices live in LDS.
//
// With 4..32 channels an offset step is a few MFMAs, so the ring kernels'
// price per step -- a barrier, a B tile through LDS, a gather's latency that
// only one other step covers -- is what they spend their time on, and below
// 32 reduction elements most of every MFMA multiplies padding.  Here the whole
// weight tensor (K x Kd x Nd, at most 110 KB) is laid out in LDS once per
// workgroup in MFMA fragment order, and from then on every wave works alone:
// it takes 16 rows of a tile, walks the tile's offsets and never meets a
// barrier.  Workgroups are persistent (as many as fit the chip) and their waves
// stride over the wave tiles, heaviest first as in the ring kernels.
//
// A step's rows come in as whole rows -- consecutive lanes take consecutive
// 16-byte chunks of a row, D steps ahead -- and pass through a per-wave LDS
// stage into the MFMA layout (a lane there holds 8 consecutive reduction
// elements of row lane % 16; loads of that shape put every lane on a cache line
// of its own and cost the address unit four times as much).  The rows' indices
// come from the tile plan a turn of four steps ahead, one load per 64 of them,
// and reach their loader lanes by shuffles.
//
// Up to 16 reduction elements, one MFMA takes several offsets: with KC =
// Kd / 8 chunks per offset rounded up to 1, 2 or 4, lane group g holds chunk
// g % KC of the step's offset g / KC, so a 16-channel layer runs two offsets
// per MFMA and a 4-channel layer four (their 16-byte rows are loaded in the
// MFMA layout as they are).  Of a step's offsets, one that no row of the 16 has
// takes a slice of zeros in its weights' place: an infinite weight reaches no
// row group that lacks its offset.  Otherwise a row sums one offset per MFMA
// in the tile's ascending order (fp32: the three products in the order of
// mfma_x3).  16-bit sums agree bitwise with the ring and pipelined kernels' at
// every width, fp32 ones from 17 elements on (below, a step's first products
// precede its second ones: the same terms, another fp32 order).
//
// Bound: at small sizes the chain head -> rows -> products of a wave tile (8 us
// with the launch up to 20,000 rows), at large ones the gathers' cache lines.
// One layer over its 27-offset map, ring / pipelined kernels before, here after:
//   4 x 16 fp32, 470,532 LiDAR voxels   69.7 -> 28.6 us
//   16 x 16 bf16, 117,000               33.5 ->  9.8 us
//   16 x 32 fp32, 4,096 uniform         24.9 ->  8.2 us
//   32 x 32 fp32, 20,001 LiDAR          24.6 -> 13.9 us
#pragma once

#include <type_traits>

#include "mfma.h"
#include "nbr_src.h"

namespace st {

constexpr int kNarrowMaxK = 64;           // a lane of a wave holds one offset of the tile's list
constexpr int kNarrowLds = 112 * 1024;    // largest weight tensor in LDS
constexpr int kNarrowLdsCu = 160 * 1024;  // LDS of a CU

constexpr int narrow_chunks(int Kd) { return Kd <= 8 ? 1 : (Kd <= 16 ? 2 : (Kd <= 32 ? 4 : 8)); }
constexpr int narrow_blocks(int Nd) { return Nd <= 16 ? 1 : (Nd <= 32 ? 2 : 4); }
// LDS bytes of the weights: per offset KC chunks x NBLK column blocks x 16 columns of 16 bytes (split fp32: two planes)
inline int64_t narrow_lds(int K, int Kd, int Nd, bool x3) {
  return (int64_t)K * narrow_chunks(Kd) * narrow_blocks(Nd) * 256 * (x3 ? 2 : 1);
}

// Whether the kernel takes a shape.  It can where rows are whole 4-element
// groups aligned to them, the arrays lie within 32-bit buffer offsets and the
// weights within the LDS.  Reductions the ring kernels are not built for (Kd
// other than 32 and 64) always come here: the alternative is the one-offset
// pipelined kernel, which was nowhere faster (here / there, us):
//                     470,532 LiDAR rows        300,000 / 900,000 indoor rows
//   fp32   16 x 64     69 / 136                  69 / 188,  258 / 491
//          20 x 32     58 / 98                   67 / 131,  272 / 353
//          40 x 16     80 / 123                 109 / 184,  390 / 495
//   16-bit  8 x 64     32 / 78                   33 / 103,  112 / 252
//          24 x 32     37 / 68                   44 / 78,   180 / 219
//          48 x 32     55 / 92                   66 / 130,  273 / 333
// At 32 and 64 the ring kernels win once the rows keep their
// larger tiles busy, so there the kernel takes sets up to a size, smaller where
// the weights fill a CU's LDS (one workgroup on a CU) and for the longer rows
// (here / ring, us, LiDAR voxels):
//   16-bit 32 x 32   117,000 rows 12.7 / 17.5   235,000 19.9 / 22.0   470,532 37.0 / 35.2
//   fp32   32 x 16   117,000      19.4 / 26.7   235,000 28.5 / 30.4   350,000 39.8 / 37.3
//   fp32   32 x 32   117,000      25.0 / 30.7   160,000 30.6 / 32.2   235,000 36.9 / 33.2
//   16-bit 64 x 16   117,000      17.5 / 20.2   160,000 20.7 / 21.8   235,000 26.6 / 24.9
//   16-bit 64 x 32    60,000      17.0 / 19.8   117,000 22.3 / 22.2   160,000 28.0 / 23.6
// An indoor set's 17 pairs a row (LiDAR: 4.7) move the crossing of 16-bit 64 x 32
// down; the other limits hold there too (whole layer, here / ring, us):
//   16-bit 64 x 32    48,000 19.9 / 24.4    90,000 31.9 / 28.7
//   16-bit 64 x 16   130,000 33.0 / 36.6    32 x 32 260,000 45.1 / 51.4    32 x 64 130,000 27.3 / 30.1
//   fp32   64 x 16    96,000 47.7 / 56.0    32 x 32 130,000 39.1 / 44.0
inline bool narrow_ok(int64_t n_src, int64_t n_dst, int K, int Kd, int Nd, size_t esz, bool x3, const void* A) {
  if (Kd > 64 || Nd > 64 || Kd % 4 != 0 || K > kNarrowMaxK) return false;
  if (narrow_chunks(Kd) * narrow_blocks(Nd) * (x3 ? 2 : 1) > 16) return false;  // not built
  if ((uintptr_t)A % (4 * esz) != 0) return false;
  if (Kd > 32 && esz == 2 && (Kd % 8 != 0 || (uintptr_t)A % 16 != 0)) return false;  // 8-byte rows: up to 32
  const int64_t lim = (1ll << 31) - 65536;  // source rows, destination rows, the plan's map (whole tiles)
  if (n_src * Kd * (int64_t)esz >= lim || n_dst * Nd * (int64_t)esz >= lim || (n_dst + 127) * K * 4 >= lim) return false;
  const int64_t lds = narrow_lds(K, Kd, Nd, x3);
  if (lds > kNarrowLds) return false;
  if ((Kd == 32 || Kd == 64) && (uintptr_t)A % 16 == 0) {
    const bool fills = 2 * lds > kNarrowLdsCu;
    if (Kd == 32) return n_dst <= (fills ? 131072 : 262144);
    return n_dst <= (fills ? (x3 ? 98304 : 65536) : 131072);
  }
  return true;
}

// 8 bytes at a byte offset of a buffer (zeros past its end).
__device__ __forceinline__ uint64_t load8(__amdgpu_buffer_rsrc_t r, int byte_offset) {
  typedef unsigned int v2u __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint64_t, __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(r, byte_offset, 0, 0)));
}

// One element at a byte offset of a buffer (zero past its end).
template <typename T>
__device__ __forceinline__ T load_elem(__amdgpu_buffer_rsrc_t r, int byte_offset) {
  if constexpr (sizeof(T) == 4)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, byte_offset, 0, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b16(r, byte_offset, 0, 0));
}

// Lays the weights out in LDS: 16-byte unit ((k * KC + q) * NBLK + nb) * PLANES
// + plane, column c, holds elements 8q .. 8q + 7 of column nb * 16 + c of slice
// k, zeros past Kd and Nd.  Whole 16-byte loads where the layout allows: along
// the reduction index from (K, Nd, Kd), eight rows of 16 bytes of columns
// transposed in registers from (K, Kd, Nd); an element at a time else.  (All
// workgroups do this once: element loads alone cost 10 us at 32 x 32.)
template <typename T, int KC, int NBLK, int NT, typename F16>
__device__ __forceinline__ void stage_weights(F16* __restrict__ w_s, const T* __restrict__ B, int b_kn, int K, int Kd,
                                              int Nd) {
  constexpr bool X3 = sizeof(T) == 4;
  constexpr int PLANES = X3 ? 2 : 1, VE = 16 / (int)sizeof(T);  // elements per 16 bytes
  typedef T vec_t __attribute__((ext_vector_type(VE)));
  const __amdgpu_buffer_rsrc_t b_rsrc = make_rsrc(B, __builtin_amdgcn_readfirstlane(K * Kd * Nd * (int)sizeof(T)));
  const bool aligned = (uintptr_t)B % 16 == 0;
  auto put = [&](int kq, int n, const T (&t)[8]) {
    F16* dst = w_s + ((kq * NBLK + n / 16) * PLANES) * 16 + n % 16;
    if constexpr (X3) {
      F16 hi, lo;
      split8(v4f{t[0], t[1], t[2], t[3]}, v4f{t[4], t[5], t[6], t[7]}, hi, lo);
      dst[0] = hi;
      dst[16] = lo;
    } else {
      F16 f;
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = t[e];
      dst[0] = f;
    }
  };
  if (b_kn && aligned && Nd % VE == 0) {
    constexpr int NV = NBLK * 16 / VE;
    for (int u = threadIdx.x; u < K * KC * NV; u += NT) {
      const int n = u % NV * VE, kq = u / NV, q = kq % KC, k = kq / KC;
      vec_t v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int kd = q * 8 + e;
        v[e] = load16<vec_t>(b_rsrc, n < Nd && kd < Kd ? ((k * Kd + kd) * Nd + n) * (int)sizeof(T) : kOobOffset);
      }
#pragma unroll
      for (int i = 0; i < VE; ++i) {
        T t[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = v[e][i];
        put(kq, n + i, t);
      }
    }
  } else if (!b_kn && aligned && Kd % VE == 0) {
#pragma unroll 4
    for (int u = threadIdx.x; u < K * KC * NBLK * 16; u += NT) {
      const int n = u % (NBLK * 16), kq = u / (NBLK * 16), q = kq % KC, k = kq / KC;
      T t[8];
#pragma unroll
      for (int h = 0; h < 8 / VE; ++h) {
        const int kd = q * 8 + h * VE;
        const vec_t v = load16<vec_t>(b_rsrc, n < Nd && kd < Kd ? ((k * Nd + n) * Kd + kd) * (int)sizeof(T) : kOobOffset);
#pragma unroll
        for (int e = 0; e < VE; ++e) t[h * VE + e] = v[e];
      }
      put(kq, n, t);
    }
  } else {
    const int se = b_kn ? Nd : 1, sn = b_kn ? 1 : Kd;  // element strides of a slice: reduction index, column
#pragma unroll 4
    for (int u = threadIdx.x; u < K * KC * NBLK * 16; u += NT) {
      const int n = u % (NBLK * 16), kq = u / (NBLK * 16), q = kq % KC, k = kq / KC;
      T t[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int kd = q * 8 + e;
        t[e] = load_elem<T>(b_rsrc, n < Nd && kd < Kd ? (k * Kd * Nd + n * sn + kd * se) * (int)sizeof(T) : kOobOffset);
      }
      put(kq, n, t);
    }
  }
}

// One element to a byte offset of a buffer (dropped past its end).
template <typename T>
__device__ __forceinline__ void store_elem(__amdgpu_buffer_rsrc_t r, int byte_offset, T v) {
  if constexpr (sizeof(T) == 4)
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), r, byte_offset, 0, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), r, byte_offset, 0, 0);
}

// T: element of A, B and out (float: split products).  KC, NBLK: chunks per
// offset and 16-column blocks.  NW: waves per workgroup.  HALF: rows are 8-byte
// aligned only (16-bit, Kd % 8 == 4).
template <typename T, int KC, int NBLK, int NW, bool HALF>
__global__ __launch_bounds__(64 * NW) void gather_gemm_narrow_kernel(const T* __restrict__ A, TiledSrc src,
                                                                     const int32_t* __restrict__ rows,
                                                                     const T* __restrict__ B, int b_kn,
                                                                     T* __restrict__ out, int n_src, int n_dst,
                                                                     int K, int Kd, int Nd, Epi<T> epi) {
  constexpr bool X3 = std::is_same<T, float>::value;
  static_assert(!(X3 && HALF), "fp32 rows are 16-byte aligned");
  using L16 = typename std::conditional<X3, __bf16, T>::type;
  using F16 = typename Frag<L16>::type;  // 8 x 16-bit MFMA operand
  constexpr int ES = (int)sizeof(T);
  constexpr int PLANES = X3 ? 2 : 1;
  constexpr int OPS = KC >= 4 ? 1 : 4 / KC;       // offsets per MFMA step
  constexpr int KS = KC > 4 ? KC / 4 : 1;         // MFMA k-steps per offset
  constexpr int D = 4;                            // row loads in flight (steps)
  constexpr int TS = 4;                           // steps per turn
  constexpr int SLICE = KC * NBLK * PLANES * 16;  // 16-byte units of weights per offset
  constexpr int ZERO = OPS > 1 ? SLICE : 0;       // a slice of zeros after the K of weights
  constexpr int WPT = kGemmBM / 16;               // wave tiles per plan tile
  constexpr int NIX = OPS;                        // index registers per turn (four offsets of 16 rows each)
  constexpr int CH = KC * (X3 ? 2 : 1);           // 16-byte chunks per source row
  constexpr int NI = OPS * 16 * CH / 64;          // row loads per step
  constexpr bool STAGED = KC > 1;
  constexpr int GR = 16 / CH > 0 ? 16 / CH : 1;   // rows per 256 bytes of the stage
  extern __shared__ __attribute__((aligned(16))) unsigned char narrow_lds_raw[];
  F16* const w_s = reinterpret_cast<F16*>(narrow_lds_raw);

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int c = lane & 15, g = lane >> 4;

  stage_weights<T, KC, NBLK, 64 * NW>(w_s, B, b_kn, K, Kd, Nd);
  for (int u = tid; u < ZERO; u += 64 * NW) w_s[K * SLICE + u] = F16{};
  __syncthreads();

  // every array through 32-bit buffer offsets (the host keeps them below 2 GB)
  const int tiles = (n_dst + kGemmBM - 1) / kGemmBM;
  const __amdgpu_buffer_rsrc_t a_rsrc = make_rsrc(A, __builtin_amdgcn_readfirstlane(n_src * Kd * ES));
  const __amdgpu_buffer_rsrc_t o_rsrc = make_rsrc(out, __builtin_amdgcn_readfirstlane(n_dst * Nd * ES));
  const __amdgpu_buffer_rsrc_t nk_rsrc = make_rsrc(src.nk, __builtin_amdgcn_readfirstlane(tiles * 4));
  const __amdgpu_buffer_rsrc_t kl_rsrc = make_rsrc(src.klist, __builtin_amdgcn_readfirstlane(tiles * K * 2));
  const __amdgpu_buffer_rsrc_t tm_rsrc = make_rsrc(src.tmap, __builtin_amdgcn_readfirstlane(tiles * K * kTileRows * 4));
  const __amdgpu_buffer_rsrc_t row_rsrc = make_rsrc(rows, __builtin_amdgcn_readfirstlane(n_dst * 4));

  const int gq = KC >= 4 ? g : g % KC, go = KC >= 4 ? 0 : g / KC;  // this lane group's chunk and offset in a step
  const F16* const w_lane = w_s + (gq * NBLK * PLANES) * 16 + c;
  // the wave's stage: chunk q of row r of the step's offset o at unit (o * 16 + r) * CH + (q ^ (r / GR % CH)):
  // stores are contiguous, and the 16 rows of a fragment read fall on 16 different 16-byte bank groups
  v4f* const st = reinterpret_cast<v4f*>(w_s + K * SLICE + ZERO) + wid * (STAGED ? NI * 64 : 0);
  // Loader lanes: load v of a step brings chunk q of row r of the step's offset o, flat = v * 64 + lane =
  // (o * 16 + r) * CH + q (not staged: the MFMA layout, chunk v of row c of offset g).  A chunk past the row's
  // end takes an offset past the buffer's.
  uint32_t l_add[NI];
  int l_from[NI];
#pragma unroll
  for (int v = 0; v < NI; ++v) {
    const int flat = v * 64 + lane, q = STAGED ? flat % CH : v;
    l_add[v] = q * 16 < Kd * ES ? q * 16 : (uint32_t)kOobOffset;
    l_from[v] = flat / CH;  // lane of the step's indices (row r of offset o at o * 16 + r)
  }

  float em[NBLK], ea[NBLK];  // the epilogue's per-column terms
#pragma unroll
  for (int nb = 0; nb < NBLK; ++nb) epi.column(nb * 16 + c, Nd, em[nb], ea[nb]);

  // Source rows of a turn's offsets: register i, lane l holds row l % 16 of offset (turn * NIX + i) * 4 + l / 16.
  // (Lanes past the tile's nk offsets read past the end: the plan reserves K offsets a tile, five times what a
  // sparse tile uses.)
  auto load_idx = [&](int wt, int turn, int nk, int32_t (&ix)[NIX]) {
    const int base = ((wt / WPT * K + turn * NIX * 4) * kTileRows + (wt % WPT) * 16) * 4;
#pragma unroll
    for (int i = 0; i < NIX; ++i)
      ix[i] = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(
          tm_rsrc, (turn * NIX + i) * 4 + g < nk ? (g * kTileRows + c) * 4 : kOobOffset, base + i * 4 * kTileRows * 4, 0);
  };
  // ... turned into byte offsets of A (past its end where there is no source), and which lanes have one
  auto to_offsets = [&](int turn, int nk, int32_t (&ix)[NIX], uint64_t (&act)[NIX]) {
#pragma unroll
    for (int i = 0; i < NIX; ++i) {
      const bool ok = (turn * NIX + i) * 4 + g < nk && (uint32_t)ix[i] < (uint32_t)n_src;
      act[i] = __ballot(ok);
      ix[i] = ok ? ix[i] * (Kd * ES) : kOobOffset;
    }
  };
  // A wave tile's offset list, indices of its first two turns and destination
  // rows, loaded a whole wave tile ahead, its offset count two ahead (scalar
  // loads would put their wait on every LDS read).
  struct Head {
    int32_t nk, k, ix[2][NIX];
    v4f drow;
  };
  auto load_nk = [&](int wt) {
    return (int32_t)__builtin_amdgcn_raw_buffer_load_b32(nk_rsrc, wt >= 0 ? 0 : kOobOffset, max(wt, 0) / WPT * 4, 0);
  };
  auto load_head = [&](int wt, int nk, Head& h) {  // (wt < 0: nothing is read)
    const int t = max(wt, 0);
    h.nk = nk;
    h.k = (int32_t)__builtin_amdgcn_raw_buffer_load_b16(kl_rsrc, lane < nk ? lane * 2 : kOobOffset, t / WPT * K * 2, 0);
    load_idx(t, 0, nk, h.ix[0]);
    load_idx(t, 1, nk, h.ix[1]);
    h.drow = load16<v4f>(row_rsrc, wt >= 0 ? (t * 16 + g * 4) * 4 : kOobOffset);  // lane group g: rows 4g .. 4g + 3
  };

  v4f raw[D][NI];  // a step's rows as loaded
  // rows of step S of the turn whose offsets are off
  auto load_rows = [&](const int32_t (&off)[NIX], auto sc) {
    constexpr int S = decltype(sc)::value, R = S * OPS / 4, L = S * OPS % 4 * 16;
#pragma unroll
    for (int v = 0; v < NI; ++v) {
      int from = off[R];
      if constexpr (STAGED) from = __shfl(from, L + l_from[v], 64);
      const uint32_t at = (uint32_t)from + l_add[v];
      if constexpr (HALF) {
        const bool second = l_add[v] + 16 <= (uint32_t)(Kd * ES);
        const uint64_t h[2] = {load8(a_rsrc, (int)at), load8(a_rsrc, second ? (int)(at + 8) : kOobOffset)};
        raw[S % D][v] = __builtin_bit_cast(v4f, h);
      } else {
        raw[S % D][v] = load16<v4f>(a_rsrc, (int)at);
      }
    }
  };

  // (a wave's index is uniform: readfirstlane lets its addresses be scalar)
  const int w0 = __builtin_amdgcn_readfirstlane((int)blockIdx.x * NW + wid);
  const int stride = (int)gridDim.x * NW;
  int wt = tiles * WPT - 1 - w0;
  if (wt < 0) return;
#define ST_IC(v) std::integral_constant<int, (v)>()
  Head cur, nxt;
  uint64_t act[NIX], actn[NIX];
  auto begin = [&]() {
    to_offsets(0, cur.nk, cur.ix[0], act);
    load_rows(cur.ix[0], ST_IC(0));
    load_rows(cur.ix[0], ST_IC(1));
    load_rows(cur.ix[0], ST_IC(2));
    load_rows(cur.ix[0], ST_IC(3));
  };
  int nk1 = load_nk(wt), nk2 = load_nk(wt - stride);
  load_head(wt, __builtin_amdgcn_readfirstlane(nk1), cur);
  load_head(wt - stride, __builtin_amdgcn_readfirstlane(nk2), nxt);
  nk2 = load_nk(wt - 2 * stride);
  begin();
  for (;;) {
    const int nk = cur.nk;
    int kreg = (src.rev ? K - 1 - cur.k : cur.k) * SLICE;  // lane j: where the weights of the j-th offset start

    v4f acc[NBLK];
#pragma unroll
    for (int nb = 0; nb < NBLK; ++nb) acc[nb] = v4f{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int j, auto sc) {
      constexpr int S = decltype(sc)::value, R = S * OPS / 4, L = S * OPS % 4 * 16;
      constexpr uint64_t lanes = OPS == 4 ? ~0ull : ((1ull << (OPS * 16)) - 1) << L;
      if (!(act[R] & lanes)) return;
      const F16* w = w_lane;
      if constexpr (OPS == 1) {
        w += __builtin_amdgcn_readlane(kreg, j);
      } else {
        const int at = __shfl(kreg, min(j * OPS + go, nk - 1), 64);
        w += (act[R] >> (L + go * 16)) & 0xffff ? at : K * SLICE;
      }
      F16 bh[KS][NBLK], bl[KS][NBLK];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int nb = 0; nb < NBLK; ++nb) {
          bh[ks][nb] = w[(ks * 4 * NBLK + nb) * PLANES * 16];
          if constexpr (X3) bl[ks][nb] = w[((ks * 4 * NBLK + nb) * PLANES + 1) * 16];
        }
      if constexpr (STAGED) {
#pragma unroll
        for (int v = 0; v < NI; ++v) {
          const int flat = v * 64 + lane, q = flat % CH, row = flat / CH;
          st[row * CH + (q ^ (row % 16 / GR % CH))] = raw[S % D][v];
        }
        // LDS operations of one wave complete in order; the fences keep the
        // compiler from moving the fragment reads above the stores, and the
        // next step's stores above the reads.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
      const v4f* const row = st + (go * 16 + c) * CH;
      const int z = c / GR % CH;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int q = ks * 4 + gq;  // chunk of 8 elements
        if constexpr (X3) {
          F16 ah, al;
          if constexpr (STAGED)
            split8(row[(2 * q) ^ z], row[(2 * q + 1) ^ z], ah, al);
          else
            split8(raw[S % D][0], raw[S % D][NI - 1], ah, al);
#pragma unroll
          for (int nb = 0; nb < NBLK; ++nb) acc[nb] = mfma_x3(ah, al, bh[ks][nb], bl[ks][nb], acc[nb]);
        } else {
          const F16 a = __builtin_bit_cast(F16, STAGED ? row[q ^ z] : raw[S % D][0]);
#pragma unroll
          for (int nb = 0; nb < NBLK; ++nb) acc[nb] = mfma(a, bh[ks][nb], acc[nb]);
        }
      }
      if constexpr (STAGED) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
    };
    // A turn: each step's products, then the same step's rows of the next turn
    // into its slot; the indices of the turn after that load meanwhile.
    const int nsteps = (nk + OPS - 1) / OPS;
    for (int j = 0, turn = 0; j < nsteps; j += TS, ++turn) {
      int32_t off[NIX];
#pragma unroll
      for (int i = 0; i < NIX; ++i) off[i] = cur.ix[1][i];
      load_idx(wt, turn + 2, nk, cur.ix[1]);
      to_offsets(turn + 1, nk, off, actn);
      multiply(j, ST_IC(0));
      load_rows(off, ST_IC(0));
      multiply(j + 1, ST_IC(1));
      load_rows(off, ST_IC(1));
      multiply(j + 2, ST_IC(2));
      load_rows(off, ST_IC(2));
      multiply(j + 3, ST_IC(3));
      load_rows(off, ST_IC(3));
#pragma unroll
      for (int i = 0; i < NIX; ++i) act[i] = actn[i];
    }

    // values first, stores after: an epilogue that reads (the residual) issues
    // all its loads before the first store, which may alias them
    int32_t drow[4];
    __builtin_memcpy(drow, &cur.drow, 16);
    float ov[4][NBLK];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int nb = 0; nb < NBLK; ++nb) {
        const int col = nb * 16 + c;
        const bool ok = wt * 16 + g * 4 + r < n_dst && col < Nd;
        // (rows past the end: row 0 of the residual, not stored)
        ov[r][nb] = epi.apply(acc[nb][r], em[nb], ea[nb], ok ? drow[r] : 0, Nd, ok ? col : 0);
      }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int at = wt * 16 + g * 4 + r < n_dst ? (drow[r] * Nd + c) * ES : kOobOffset;
#pragma unroll
      for (int nb = 0; nb < NBLK; ++nb)
        store_elem<T>(o_rsrc, nb * 16 + c < Nd ? at + nb * 16 * ES : kOobOffset, from_f32<T>(ov[r][nb]));
    }
    // The next wave tile's first gathers, its head here since the last one; the
    // head after it goes out before them: memory answers in order, so the wait
    // for those gathers is the wait for it as well.
    wt -= stride;
    if (wt < 0) break;
    cur = nxt;
    load_head(wt - stride, __builtin_amdgcn_readfirstlane(nk2), nxt);
    nk2 = load_nk(wt - 2 * stride);
    begin();
  }
#undef ST_IC
}

template <typename T, int KC, int NBLK, bool HALF>
static void launch_narrow_shape(const T* A, int64_t n_src, const TiledSrc& src, const int32_t* rows, const T* B,
                                int b_kn, T* out, Epi<T> epi, int64_t n_dst, int K, int Kd, int Nd,
                                hipStream_t stream) {
  constexpr int STAGE = KC > 1 ? (KC >= 4 ? 1 : 4 / KC) * 16 * KC * (sizeof(T) == 4 ? 2 : 1) * 16 : 0;  // bytes per wave
  const int w_lds = (int)narrow_lds(K + (KC < 4), Kd, Nd, sizeof(T) == 4);  // (up to 16 elements: and the slice of zeros)
  const int64_t wave_tiles = (n_dst + kGemmBM - 1) / kGemmBM * (kGemmBM / 16);
  auto launch = [&](auto nw) {
    constexpr int NW = decltype(nw)::value;
    const int64_t need = (wave_tiles + NW - 1) / NW;
    const int lds = w_lds + NW * STAGE, fit = kNarrowLdsCu / lds, most = 256 * (fit < 32 / NW ? fit : 32 / NW);
    gather_gemm_narrow_kernel<T, KC, NBLK, NW, HALF><<<(unsigned)(need < most ? need : most), 64 * NW, lds, stream>>>(
        A, src, rows, B, b_kn, out, (int)n_src, (int)n_dst, K, Kd, Nd, epi);
  };
  // Eight waves a workgroup, as many workgroups as 32 waves a CU and the LDS
  // hold; sixteen where the weights leave room for one workgroup on a CU, once
  // the rows fill more than one workgroup of eight on every CU.
  if (KC * NBLK * sizeof(T) >= 32 && STAGE <= 2048 && kNarrowLdsCu / (w_lds + 8 * STAGE) < 2 && wave_tiles > 256 * 8)
    launch(std::integral_constant<int, 16>());
  else
    launch(std::integral_constant<int, 8>());
}

// Launches the kernel for a shape narrow_ok accepts.
template <typename T>
static void launch_narrow(const T* A, int64_t n_src, const TiledSrc& src, const int32_t* rows, const T* B, int b_kn,
                          T* out, Epi<T> epi, int64_t n_dst, int K, int Kd, int Nd, hipStream_t stream) {
  const int kc = narrow_chunks(Kd), nb = narrow_blocks(Nd);
  const bool half = sizeof(T) == 2 && (Kd % 8 != 0 || (uintptr_t)A % 16 != 0);
#define ST_NARROW(KC_, NB_)                                                                                          \
  if (kc == KC_ && nb == NB_) {                                                                                      \
    if constexpr (sizeof(T) == 2 && KC_ <= 4) {                                                                      \
      if (half) {                                                                                                    \
        launch_narrow_shape<T, KC_, NB_, true>(A, n_src, src, rows, B, b_kn, out, epi, n_dst, K, Kd, Nd, stream);    \
        return;                                                                                                      \
      }                                                                                                              \
    }                                                                                                                \
    if constexpr (KC_ * NB_ * sizeof(T) <= 32)                                                                       \
      launch_narrow_shape<T, KC_, NB_, false>(A, n_src, src, rows, B, b_kn, out, epi, n_dst, K, Kd, Nd, stream);     \
  }
  ST_NARROW(1, 1) ST_NARROW(1, 2) ST_NARROW(1, 4) ST_NARROW(2, 1) ST_NARROW(2, 2) ST_NARROW(2, 4)
  ST_NARROW(4, 1) ST_NARROW(4, 2) ST_NARROW(4, 4) ST_NARROW(8, 1) ST_NARROW(8, 2)
#undef ST_NARROW
}

}  // namespace st
