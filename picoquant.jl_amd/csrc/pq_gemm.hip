// Complex GEMM on CDNA4 matrix cores with the index permutation fused into
// operand loads and result stores (TTGT without the transposes).
//
//   C[m, n] = sum_k A[m, k] * B[k, n]      (per batch entry z)
//
// m, n, k are linear indices of the M / N / K index groups; element offsets
// come from per-workgroup offset tables in LDS (row tables for the tile,
// K tables in windows of 1024), so any stride pattern is read and written
// in place.
//
// Complex product as four real MFMAs on split planes:
//   Cr += Ar*Br + (-Ai)*Bi ;  Ci += Ar*Bi + Ai*Br
// complex64  -> v_mfma_f32_16x16x4_f32 (fp32 accumulate)
// complex128 -> v_mfma_f64_16x16x4_f64 (fp64 accumulate)
//
// Tile: 256 lanes = 4 waves arranged WGM x WGN (2x2, 4x1 or 1x4); workgroup
// tile BM x BN, each wave (BM/WGM) x (BN/WGN) as a grid of 16x16 MFMA tiles.
// Extents below the tile are zero-padded.  Lane layout of a 16x16x4 MFMA (64 lanes): A operand lane l holds
// A[l%16][l/16], B operand B[l/16][l%16]; accumulator register r holds
// D[4*(l/16)+r][l%16] for f32 and D[l/16+4r][l%16] for f64.
#include "pq_internal.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

template <typename R> struct mfma_t;
template <> struct mfma_t<float> {
  typedef floatx4 acc;
  // accumulator register r of lane-group g (= lane/16) holds row 4*g + r
  static __device__ __forceinline__ int row(int g, int r) { return 4 * g + r; }
  static __device__ __forceinline__ acc op(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};
template <> struct mfma_t<double> {
  typedef doublex4 acc;
  // the f64 variant interleaves: register r of lane-group g holds row g + 4*r
  static __device__ __forceinline__ int row(int g, int r) { return g + 4 * r; }
  static __device__ __forceinline__ acc op(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};

constexpr int KTAB_MAX = 1024;   // K offsets that k_gemm holds in LDS at a time
constexpr uint32_t GEMM_K_MAX = 1u << 24;

// Workgroups are dealt to the 8 XCDs round-robin in launch order, and each
// XCD has its own L2.  Renumber the (x, y) tiles of a batch entry so that
// each XCD gets one contiguous run of tiles: the tiles that share rows of
// the large operand (consecutive x for one y) then meet in the same L2.
__device__ __forceinline__ void xcd_tile(uint32_t& tx, uint32_t& ty) {
  const uint32_t gx = gridDim.x, n = gridDim.x * gridDim.y;
  const uint32_t b = blockIdx.x + gx * blockIdx.y;
  uint32_t l = b;
  if (n % 8 == 0 && n >= 16) l = (b % 8) * (n / 8) + b / 8;
  tx = l % gx;
  ty = l / gx;
}

// FP32 accumulation in two levels: each K tile's products are summed in a
// fresh accumulator (at most 16 MFMA roundings), which is then added to the
// running sum.  A single chain over K = 256 rounds 128 times into a growing
// sum; two levels cut the rounding error of long sums about 2-3x for 2x the
// accumulator registers.  FP64 accumulates in one chain.
template <typename MF, int TM, int TN>
__device__ __forceinline__ void zero_acc(typename MF::acc (&xr)[TM][TN], typename MF::acc (&xi)[TM][TN]) {
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        xr[i][j][r] = 0;
        xi[i][j][r] = 0;
      }
}

template <typename MF, int TM, int TN>
__device__ __forceinline__ void add_chunk(typename MF::acc (&accr)[TM][TN], typename MF::acc (&acci)[TM][TN],
                                          const typename MF::acc (&cr)[TM][TN], const typename MF::acc (&ci)[TM][TN]) {
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        accr[i][j][r] += cr[i][j][r];
        acci[i][j][r] += ci[i][j][r];
      }
}

// One K step (4 values of K) of a wave's TM x TN complex blocks; fresh: the
// sums start at zero.  Each real product runs over all blocks before the
// next one, so consecutive MFMAs never wait for each other's accumulator.
template <typename MF, int TM, int TN, typename C>
__device__ __forceinline__ void mfma_step(typename MF::acc (&xr)[TM][TN], typename MF::acc (&xi)[TM][TN],
                                          const C (&a)[TM], const C (&b)[TN], bool fresh) {
  const typename MF::acc zero = {};
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) xr[i][j] = MF::op(a[i].x, b[j].x, fresh ? zero : xr[i][j]);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) xi[i][j] = MF::op(a[i].x, b[j].y, fresh ? zero : xi[i][j]);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) xr[i][j] = MF::op(-a[i].y, b[j].y, xr[i][j]);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) xi[i][j] = MF::op(a[i].y, b[j].x, xi[i][j]);
}

// ------------------------------------------------------------------- k_gemm
// Any stride pattern.  Element offsets are row offset + K offset: each
// lane's row offsets stay in registers, the K offsets of a window of
// KTAB_MAX indices in an LDS table.  The next K tile's elements are gathered
// into registers while the matrix cores work on the current one, and LDS
// holds interleaved complex values at an odd pitch, as in k_gemm2 (whose
// main loop this is).
// Bound: MFMA (79 % busy on a 2^13 x 2^9 x 2^11 complex64 product with every
// index order shuffled; operands with unit stride along M and N take the same
// time, so the gather is hidden).  That product: 738 us loading, storing and
// multiplying each K tile in turn, 566 us with the register prefetch, 552 us
// with each real product issued over all blocks; 2^11 x 2^7 x 2^9 complex128
// 23.2 -> 16.8 us (calls overlapped on three streams).  K tiles of 32 take
// the same time within 2 % and round more (longer first-level sums).
template <typename C, int BM, int BN, int WGM, bool AK, bool BK_FAST>
__global__ __launch_bounds__(256) void k_gemm(const C* __restrict__ A, const C* __restrict__ B,
                                              C* __restrict__ Out, GemmArgs g) {
  typedef typename real_of<C>::type R;
  typedef mfma_t<R> MF;
  constexpr int WGN = 4 / WGM;
  constexpr int WM = BM / WGM, WN = BN / WGN;    // wave tile
  static_assert(WM % 16 == 0 && WN % 16 == 0, "wave tile must be a multiple of 16");
  constexpr int BKT = 16;                        // K tile
  constexpr int TM = WM / 16, TN = WN / 16;      // 16x16 tiles per wave
  constexpr bool CHUNKED = sizeof(R) == 4;
  constexpr int LDK = BKT + 1;                   // LDS row pitch (complex elements)
  constexpr int ANE = BM * BKT / 256, BNE = BN * BKT / 256;   // elements per lane of each tile

  __shared__ C As[BM * LDK], Bs[BN * LDK];
  __shared__ int32_t offCm[BM], offCn[BN];
  __shared__ int32_t offAm[BM], offBn[BN];
  __shared__ int32_t offAk[KTAB_MAX], offBk[KTAB_MAX];

  PQ_TOUCH(g.M, g.N, g.K, g.L);
  const uint32_t Mt = g.M.total, Nt = g.N.total, Kt = g.K.total;
  uint32_t tile_x, tile_y;
  xcd_tile(tile_x, tile_y);
  const uint32_t m0 = tile_x * BM, n0 = tile_y * BN;
  const int tid = threadIdx.x;
  {
    int64_t oa, ob, oc;
    batch_offsets(g.L, blockIdx.z, oa, ob, oc);
    A += oa;
    B += ob;
    Out += oc;
  }

  // rows past an operand's extent read its first row; their products only
  // reach outputs that are never stored
  for (int t = tid; t < BM + BN; t += 256) {
    int32_t o = 0, oc = 0;
    if (t < BM) {
      if (m0 + t < Mt) group_offsets(g.M, m0 + t, o, oc);
      offAm[t] = o;
      offCm[t] = oc;
    } else {
      if (n0 + t - BM < Nt) group_offsets(g.N, n0 + t - BM, o, oc);
      offBn[t - BM] = o;
      offCn[t - BM] = oc;
    }
  }
  // K offsets of the window that starts at kb (entries past K: offset 0,
  // zeroed when the tile is stored)
  auto fill_window = [&](uint32_t kb) {
    for (uint32_t t = tid; t < (uint32_t)KTAB_MAX && t < Kt - kb + BKT; t += 256) {
      int32_t oa = 0, ob = 0;
      if (kb + t < Kt) group_offsets(g.K, kb + t, oa, ob);
      offAk[t] = oa;
      offBk[t] = ob;
    }
  };
  fill_window(0);
  __syncthreads();

  // This lane's elements of a tile: with the lanes along K, one K index and
  // every 256 / BKT-th row; else every 256 / BM-th K index of one row
  // (BM = 256 / BKT rows or more; a narrower tile's lanes wrap).
  const int ak = AK ? tid % BKT : tid / BM, am = AK ? tid / BKT : tid % BM;
  const int bk = BK_FAST ? tid % BKT : tid / BN, bn = BK_FAST ? tid / BKT : tid % BN;
  constexpr int AKS = AK ? 0 : 256 / BM, AMS = AK ? 256 / BKT : 0;   // step per element
  constexpr int BKS = BK_FAST ? 0 : 256 / BN, BNS = BK_FAST ? 256 / BKT : 0;
  int32_t ga[AK ? ANE : 1], gb[BK_FAST ? BNE : 1];
#pragma unroll
  for (int q = 0; q < (AK ? ANE : 1); ++q) ga[q] = offAm[am + AMS * q];
#pragma unroll
  for (int q = 0; q < (BK_FAST ? BNE : 1); ++q) gb[q] = offBn[bn + BNS * q];

  const int wave = tid / 64, lane = tid % 64;
  const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;
  const int li = lane % 16, lk = lane / 16;

  typename MF::acc accr[TM][TN], acci[TM][TN];
  zero_acc<MF, TM, TN>(accr, acci);

  C ra[ANE], rb[BNE];
  auto load_tile = [&](uint32_t k0) {            // k0: the tile's place in the window
#pragma unroll
    for (int q = 0; q < ANE; ++q) ra[q] = A[ga[AK ? q : 0] + offAk[k0 + ak + AKS * q]];
#pragma unroll
    for (int q = 0; q < BNE; ++q) rb[q] = B[gb[BK_FAST ? q : 0] + offBk[k0 + bk + BKS * q]];
  };
  auto store_tile = [&](uint32_t left) {         // left: K values from this tile on
    if (left < (uint32_t)BKT) {
#pragma unroll
      for (int q = 0; q < ANE; ++q)
        if ((uint32_t)(ak + AKS * q) >= left) ra[q].x = ra[q].y = 0;
#pragma unroll
      for (int q = 0; q < BNE; ++q)
        if ((uint32_t)(bk + BKS * q) >= left) rb[q].x = rb[q].y = 0;
    }
#pragma unroll
    for (int q = 0; q < ANE; ++q) As[(am + AMS * q) * LDK + ak + AKS * q] = ra[q];
#pragma unroll
    for (int q = 0; q < BNE; ++q) Bs[(bn + BNS * q) * LDK + bk + BKS * q] = rb[q];
  };

  const C* Ap = As + (wm + li) * LDK + lk;
  const C* Bp = Bs + (wn + li) * LDK + lk;
  load_tile(0);
  for (uint32_t k0 = 0; k0 < Kt; k0 += BKT) {
    typename MF::acc cr[TM][TN], ci[TM][TN];
    store_tile(Kt - k0);
    __syncthreads();
    if (k0 + BKT < Kt) {
      const uint32_t next = (k0 + BKT) % KTAB_MAX;
      if (next == 0) {
        // past the barrier every lane has read its offsets of this window
        fill_window(k0 + BKT);
        __syncthreads();
      }
      load_tile(next);
    }
#pragma unroll
    for (int kk = 0; kk < BKT; kk += 4) {
      C a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = Ap[16 * i * LDK + kk];
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j] = Bp[16 * j * LDK + kk];
      // a K tile's first products start the tile's fresh sums
      if constexpr (CHUNKED)
        mfma_step<MF, TM, TN>(cr, ci, a, b, kk == 0);
      else
        mfma_step<MF, TM, TN>(accr, acci, a, b, false);
    }
    if constexpr (CHUNKED) add_chunk<MF, TM, TN>(accr, acci, cr, ci);
    __syncthreads();
  }

  // Epilogue: accumulator register r of tile (i, j) holds D[MF::row(lk, r)][li].
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        int m = wm + 16 * i + MF::row(lk, r);
        int n = wn + 16 * j + li;
        if (m0 + m < Mt && n0 + n < Nt) {
          C v;
          v.x = accr[i][j][r];
          v.y = acci[i][j][r];
          Out[offCm[m] + offCn[n]] = v;
        }
      }
}

// ------------------------------------------------------------------ k_gemm2
// Fast path when the summed indices run contiguously in both operands
// (first K mode has unit stride in A and in B and its extent is a multiple
// of BKT) and every offset keeps 16-byte alignment: each operand row (A) or
// column (B) of a K tile is one contiguous run, read with 16-byte vector
// loads.  The next tile is prefetched into registers while the matrix
// cores work on the current one (register double buffering).
//
// LDS holds the tiles as interleaved complex values, row-major [row][k]
// with an odd pitch of BKT + 1 elements: a lane's (re, im) operand pair is
// one 8-byte (16-byte for complex128) read, and the 16 lanes of an MFMA
// operand row fall on distinct banks.
template <typename C, int BM, int BN, int WGM, int BKT>
__global__ __launch_bounds__(256) void k_gemm2(const C* __restrict__ A, const C* __restrict__ B,
                                               C* __restrict__ Out, GemmArgs g) {
  typedef typename real_of<C>::type R;
  typedef mfma_t<R> MF;
  constexpr int WGN = 4 / WGM;
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int TM = WM / 16, TN = WN / 16;
  static_assert(WM % 16 == 0 && WN % 16 == 0, "wave tile must be a multiple of 16");
  constexpr bool CHUNKED = sizeof(R) == 4;
  constexpr int VEC = 16 / (int)sizeof(C);       // complex elements per 16-byte chunk
  constexpr int CPR = BKT / VEC;                  // chunks per row of a K tile
  constexpr int ACH = (BM * CPR + 255) / 256;     // chunks per lane, A tile
  constexpr int BCH = (BN * CPR + 255) / 256;     // chunks per lane, B tile
  constexpr int KT_MAX = 2048 / BKT;              // K tiles (K <= 2048)
  constexpr int LDK = BKT + 1;                    // LDS row pitch (complex elements)

  __shared__ C As[BM * LDK + VEC];   // + a spare chunk written by idle lanes
  __shared__ C Bs[BN * LDK + VEC];
  __shared__ int32_t offAm[BM], offCm[BM], offBn[BN], offCn[BN];
  __shared__ int32_t offAk[KT_MAX], offBk[KT_MAX];

  PQ_TOUCH(g.M, g.N, g.K, g.L);
  const uint32_t Mt = g.M.total, Nt = g.N.total, Kt = g.K.total;
  uint32_t tile_x, tile_y;
  xcd_tile(tile_x, tile_y);
  const uint32_t m0 = tile_x * BM, n0 = tile_y * BN;
  const int tid = threadIdx.x;
  {
    int64_t oa, ob, oc;
    batch_offsets(g.L, blockIdx.z, oa, ob, oc);
    A += oa;
    B += ob;
    Out += oc;
  }
  for (int t = tid; t < BM; t += 256) {
    int32_t oa = 0, oc = 0;
    if (m0 + t < Mt) group_offsets(g.M, m0 + t, oa, oc);
    offAm[t] = oa;
    offCm[t] = oc;
  }
  for (int t = tid; t < BN; t += 256) {
    int32_t ob = 0, oc = 0;
    if (n0 + t < Nt) group_offsets(g.N, n0 + t, ob, oc);
    offBn[t] = ob;
    offCn[t] = oc;
  }
  // K tile offsets: a table when the tiles fit it, else decoded per tile
  // (the same value in every lane)
  const uint32_t ntiles = Kt / BKT;
  const bool ktab = ntiles <= (uint32_t)KT_MAX;
  if (ktab) {
    for (uint32_t t = tid; t < ntiles; t += 256) {
      int32_t oa, ob;
      group_offsets(g.K, t * BKT, oa, ob);
      offAk[t] = oa;
      offBk[t] = ob;
    }
  }
  __syncthreads();

  // This lane's chunks of each tile: global offset (fixed over K) and LDS
  // position.  Loads and stores are unconditional: rows past the operand's
  // extent read its first row (offAm / offBn hold 0 there), and their
  // products only reach outputs that are never stored; lanes past the tile
  // (when 256 does not divide its chunk count) write a spare LDS chunk.
  int32_t ga[ACH], gb[BCH], la[ACH], lb[BCH];
#pragma unroll
  for (int q = 0; q < ACH; ++q) {
    const int id = tid + 256 * q;
    const int row = id / CPR, cc = id % CPR;
    ga[q] = (row < BM ? offAm[row] : 0) + cc * VEC;
    la[q] = row < BM ? row * LDK + cc * VEC : BM * LDK;
  }
#pragma unroll
  for (int q = 0; q < BCH; ++q) {
    const int id = tid + 256 * q;
    const int col = id / CPR, cc = id % CPR;
    gb[q] = (col < BN ? offBn[col] : 0) + cc * VEC;
    lb[q] = col < BN ? col * LDK + cc * VEC : BN * LDK;
  }

  const int wave = tid / 64, lane = tid % 64;
  const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;
  const int li = lane % 16, lk = lane / 16;

  typename MF::acc accr[TM][TN], acci[TM][TN];
  zero_acc<MF, TM, TN>(accr, acci);

  // 16-byte staging registers: two complex64 or one complex128 per chunk
  typedef typename std::conditional<sizeof(C) == 8, float4, double2>::type V16;
  V16 ra[ACH], rb[BCH];
  auto load_tile = [&](uint32_t kt) {
    int32_t ka, kb;
    if (ktab) {
      ka = offAk[kt];
      kb = offBk[kt];
    } else {
      group_offsets(g.K, kt * BKT, ka, kb);
    }
#pragma unroll
    for (int q = 0; q < ACH; ++q) ra[q] = *reinterpret_cast<const V16*>(A + ga[q] + ka);
#pragma unroll
    for (int q = 0; q < BCH; ++q) rb[q] = *reinterpret_cast<const V16*>(B + gb[q] + kb);
  };
  auto put = [](C* dst, const V16& v) {
    if constexpr (VEC == 2) {
      C x, y;
      x.x = v.x;
      x.y = v.y;
      y.x = v.z;
      y.y = v.w;
      dst[0] = x;
      dst[1] = y;
    } else {
      C x;
      x.x = v.x;
      x.y = v.y;
      dst[0] = x;
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int q = 0; q < ACH; ++q) put(As + la[q], ra[q]);
#pragma unroll
    for (int q = 0; q < BCH; ++q) put(Bs + lb[q], rb[q]);
  };

  const C* Ap = As + (wm + li) * LDK + lk;
  const C* Bp = Bs + (wn + li) * LDK + lk;
  load_tile(0);
  for (uint32_t kt = 0; kt < ntiles; ++kt) {
    typename MF::acc cr[TM][TN], ci[TM][TN];
    store_tile();
    __syncthreads();
    if (kt + 1 < ntiles) load_tile(kt + 1);
#pragma unroll
    for (int kk = 0; kk < BKT; kk += 4) {
      C a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = Ap[16 * i * LDK + kk];
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j] = Bp[16 * j * LDK + kk];
      // a K tile's first products start the tile's fresh sums
      if constexpr (CHUNKED)
        mfma_step<MF, TM, TN>(cr, ci, a, b, kk == 0);
      else
        mfma_step<MF, TM, TN>(accr, acci, a, b, false);
    }
    if constexpr (CHUNKED) add_chunk<MF, TM, TN>(accr, acci, cr, ci);
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        int m = wm + 16 * i + MF::row(lk, r);
        int n = wn + 16 * j + li;
        if (m0 + m < Mt && n0 + n < Nt) {
          C v;
          v.x = accr[i][j][r];
          v.y = acci[i][j][r];
          Out[offCm[m] + offCn[n]] = v;
        }
      }
}

// K-tile depth of the fast path: 32 for complex64 tiles whose LDS allows it.
template <typename C, int BM, int BN>
constexpr int fast_bk() {
  // 32 when both tiles at pitch 33 plus the offset tables fit 80 KiB (two
  // workgroups per CU's 160 KiB); 64-deep tiles measured slower (their
  // staging registers halve the occupancy)
  constexpr size_t es = sizeof(C), tab = 16 * (BM + BN) + 2 * 4 * 2048 / 8;
  return (BM + BN + 2) * 33 * es + tab <= 80 * 1024 ? 32 : 16;
}

// Static LDS stays within 64 KiB: complex128 tiles up to 128 rows or
// columns and 4096 elements.
template <typename C, int BM, int BN>
constexpr bool tile_fits() {
  return sizeof(C) == 8 || (BM * BN <= 64 * 64 && BM <= 128 && BN <= 128);
}

template <typename C, int BM, int BN, int WGM>
hipError_t launch_tile(const C* A, const C* B, C* Out, const GemmArgs& g, hipStream_t s) {
  if constexpr (!tile_fits<C, BM, BN>()) {
    return launch_tile<C, (BM > 64 ? 64 : BM), (BN > 64 ? 64 : BN), WGM>(A, B, Out, g, s);
  } else {
    dim3 grid((g.M.total + BM - 1) / BM, (g.N.total + BN - 1) / BN, g.L.total);
    constexpr int BKF = fast_bk<C, BM, BN>();
    // K tile depth: the deepest of 32 / 16 / 8 (within the tile's LDS
    // budget) that divides the first (contiguous) K mode, so a tile never
    // straddles two runs.
    const uint32_t k0ext = g.K.nmodes > 0 ? g.K.m[0].ext.d : 0;
    if (g.contig && k0ext > 0) {
      if (k0ext % BKF == 0) {
        hipLaunchKernelGGL((k_gemm2<C, BM, BN, WGM, BKF>), grid, dim3(256), 0, s, A, B, Out, g);
        return hipGetLastError();
      }
      if (BKF > 16 && k0ext % 16 == 0) {
        hipLaunchKernelGGL((k_gemm2<C, BM, BN, WGM, 16>), grid, dim3(256), 0, s, A, B, Out, g);
        return hipGetLastError();
      }
      if (k0ext % 8 == 0) {
        hipLaunchKernelGGL((k_gemm2<C, BM, BN, WGM, 8>), grid, dim3(256), 0, s, A, B, Out, g);
        return hipGetLastError();
      }
    }
    if (g.a_kfast && g.b_kfast)
      hipLaunchKernelGGL((k_gemm<C, BM, BN, WGM, true, true>), grid, dim3(256), 0, s, A, B, Out, g);
    else if (g.a_kfast)
      hipLaunchKernelGGL((k_gemm<C, BM, BN, WGM, true, false>), grid, dim3(256), 0, s, A, B, Out, g);
    else if (g.b_kfast)
      hipLaunchKernelGGL((k_gemm<C, BM, BN, WGM, false, true>), grid, dim3(256), 0, s, A, B, Out, g);
    else
      hipLaunchKernelGGL((k_gemm<C, BM, BN, WGM, false, false>), grid, dim3(256), 0, s, A, B, Out, g);
    return hipGetLastError();
  }
}

// ----------------------------------------------------------------- k_gemm_h
// complex64 GEMM on FP16 matrix cores with a hi/lo split (the fast path's
// contiguous-K layout; K tiles of 32).  Per K tile every row of A (column of
// B) gets a power-of-two scale 2^s that brings its largest magnitude into
// [2^14, 2^15); each scaled FP32 value x is split into hi = fp16(x) and
// lo = fp16(x - hi), and the product is summed as hi*hi + hi*lo + lo*hi
// (lo*lo dropped, about 2^-22 relative) on v_mfma_f32_16x16x32_f16 with FP32
// accumulation: 12 FP16 MFMAs per 16x16 complex block and K tile.  The
// tile's sums are unscaled exactly (ldexp) and added to the running FP32
// sums, as in the FP32 path's two-level accumulation.
//
// MFMA 16x16x32 f16 lane layout (64 lanes): A lane l holds A[l%16][8(l/16)+i],
// B lane l holds B[8(l/16)+i][l%16], accumulator r holds D[4(l/16)+r][l%16].
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));

// Two values rounded to fp16, in one word, and what the rounding left of
// them (exact: x - fp16(x), the word's halves read in place).
__device__ __forceinline__ uint32_t pack16(const floatx2& x) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, half2v));
}
__device__ __forceinline__ floatx2 rest16(uint32_t h, const floatx2& x) {
  floatx2 r;
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r.x) : "v"(h), "v"(x.x));
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r.y) : "v"(h), "v"(x.y));
  return r;
}

__device__ __forceinline__ floatx4 mfma16(const half8& a, const half8& b, const floatx4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

template <int BM, int BN, int WGM>
__global__ __launch_bounds__(256) void k_gemm_h(const c64* __restrict__ A, const c64* __restrict__ B,
                                                c64* __restrict__ Out, GemmArgs g) {
  constexpr int BKT = 32;                         // complex K per tile = one MFMA depth
  constexpr int WGN = 4 / WGM;
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int TM = WM / 16, TN = WN / 16;
  static_assert(WM % 16 == 0 && WN % 16 == 0, "wave tile must be a multiple of 16");
  constexpr int CPR = BKT / 4;                    // 32-byte units (4 complex) per row
  constexpr int ACH = (BM * CPR + 255) / 256;
  constexpr int BCH = (BN * CPR + 255) / 256;
  constexpr int KT_MAX = 2048 / BKT;
  constexpr int PK = BKT + 8;                     // plane pitch in halves (16-byte aligned rows)

  // planes: 0 re-hi, 1 re-lo, 2 im-hi, 3 im-lo; one spare row for idle lanes
  __shared__ __align__(16) _Float16 Ap[4][(BM + 1) * PK];
  __shared__ __align__(16) _Float16 Bp[4][(BN + 1) * PK];
  __shared__ __align__(16) int32_t sA[BM + 1], sB[BN + 1];
  __shared__ int32_t offAm[BM], offCm[BM], offBn[BN], offCn[BN];
  __shared__ int32_t offAk[KT_MAX], offBk[KT_MAX];

  PQ_TOUCH(g.M, g.N, g.K, g.L);
  const uint32_t Mt = g.M.total, Nt = g.N.total, Kt = g.K.total;
  uint32_t tile_x, tile_y;
  xcd_tile(tile_x, tile_y);
  const uint32_t m0 = tile_x * BM, n0 = tile_y * BN;
  const int tid = threadIdx.x;
  {
    int64_t oa, ob, oc;
    batch_offsets(g.L, blockIdx.z, oa, ob, oc);
    A += oa;
    B += ob;
    Out += oc;
  }
  for (int t = tid; t < BM; t += 256) {
    int32_t oa = 0, oc = 0;
    if (m0 + t < Mt) group_offsets(g.M, m0 + t, oa, oc);
    offAm[t] = oa;
    offCm[t] = oc;
  }
  for (int t = tid; t < BN; t += 256) {
    int32_t ob = 0, oc = 0;
    if (n0 + t < Nt) group_offsets(g.N, n0 + t, ob, oc);
    offBn[t] = ob;
    offCn[t] = oc;
  }
  const uint32_t ntiles = Kt / BKT;
  const bool ktab = ntiles <= (uint32_t)KT_MAX;
  if (ktab) {
    for (uint32_t t = tid; t < ntiles; t += 256) {
      int32_t oa, ob;
      group_offsets(g.K, t * BKT, oa, ob);
      offAk[t] = oa;
      offBk[t] = ob;
    }
  }
  __syncthreads();

  // Lane units: 8 consecutive lanes hold the 8 units of one row, so a row's
  // scale is a maximum over half a DPP row.  Rows past the operand read its
  // first row; lanes past the tile use the spare row.
  int32_t ga[ACH], gb[BCH], la[ACH], lb[BCH], ra_row[ACH], rb_row[BCH];
#pragma unroll
  for (int q = 0; q < ACH; ++q) {
    const int id = tid + 256 * q;
    const int row = id / CPR, cc = id % CPR;
    ga[q] = (row < BM ? offAm[row] : 0) + cc * 4;
    ra_row[q] = row < BM ? row : BM;
    la[q] = ra_row[q] * PK + cc * 4;
  }
#pragma unroll
  for (int q = 0; q < BCH; ++q) {
    const int id = tid + 256 * q;
    const int col = id / CPR, cc = id % CPR;
    gb[q] = (col < BN ? offBn[col] : 0) + cc * 4;
    rb_row[q] = col < BN ? col : BN;
    lb[q] = rb_row[q] * PK + cc * 4;
  }
  const bool lead = (tid % CPR) == 0;

  const int wave = tid / 64, lane = tid % 64;
  const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;
  const int li = lane % 16, lk = lane / 16;

  floatx4 accr[TM][TN], acci[TM][TN];
  zero_acc<mfma_t<float>, TM, TN>(accr, acci);

  floatx4 ra[ACH][2], rb[BCH][2];
  auto load_tile = [&](uint32_t kt) {
    int32_t ka, kb;
    if (ktab) {
      ka = offAk[kt];
      kb = offBk[kt];
    } else {
      group_offsets(g.K, kt * BKT, ka, kb);
    }
#pragma unroll
    for (int q = 0; q < ACH; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h) ra[q][h] = *reinterpret_cast<const floatx4*>(A + ga[q] + ka + 2 * h);
#pragma unroll
    for (int q = 0; q < BCH; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h) rb[q][h] = *reinterpret_cast<const floatx4*>(B + gb[q] + kb + 2 * h);
  };
  // Scale of a row: 2^s brings its largest magnitude into [2^14, 2^15).
  // Magnitudes compare as integers; the maximum over the row's 8 lanes takes
  // three DPP steps.  (Through the LDS crossbar, four steps that each waited
  // for the last per 2 complex, and with every rounded value converted twice,
  // the conversion was 433 instructions per K tile; 64 x 262144 x 64 took
  // 79.4 us, now 57.5 against 52.6 at the copy rate, 64 x 32768 x 512 62.8,
  // now 41.8.)
  auto scale_of = [](const floatx4 (&v)[2]) {
    uint32_t m = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = v[h][r];
        m = max(m, __builtin_bit_cast(uint32_t, x) & 0x7fffffffu);
      }
    m = max(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x141, 0xf, 0xf, true));   // l and 7 - l
    m = max(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x4e, 0xf, 0xf, true));    // quad 2, 3, 0, 1
    m = max(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0xb1, 0xf, 0xf, true));    // quad 1, 0, 3, 2
    int e = 0;
    (void)frexpf(__builtin_bit_cast(float, m), &e);
    return m != 0 ? 15 - e : 0;
  };
  // Splits and stores one unit (4 complex) of a row into the planes.
  auto split_store = [&](_Float16* p0, _Float16* p1, _Float16* p2, _Float16* p3, int at, const floatx4 (&v)[2],
                         int sc) {
    uint2v hr, lr, hi, lo;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      floatx2 x, y;
      x.x = ldexpf(v[h][0], sc);
      y.x = ldexpf(v[h][1], sc);
      x.y = ldexpf(v[h][2], sc);
      y.y = ldexpf(v[h][3], sc);
      hr[h] = pack16(x);
      hi[h] = pack16(y);
      lr[h] = pack16(rest16(hr[h], x));
      lo[h] = pack16(rest16(hi[h], y));
    }
    *reinterpret_cast<uint2v*>(p0 + at) = hr;
    *reinterpret_cast<uint2v*>(p1 + at) = lr;
    *reinterpret_cast<uint2v*>(p2 + at) = hi;
    *reinterpret_cast<uint2v*>(p3 + at) = lo;
  };
  auto negate = [](const half8& x) {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(half8, __builtin_bit_cast(u4, x) ^ 0x80008000u);
  };

  load_tile(0);
  for (uint32_t kt = 0; kt < ntiles; ++kt) {
    int ea[ACH], eb[BCH];
#pragma unroll
    for (int q = 0; q < ACH; ++q) ea[q] = scale_of(ra[q]);
#pragma unroll
    for (int q = 0; q < BCH; ++q) eb[q] = scale_of(rb[q]);
#pragma unroll
    for (int q = 0; q < ACH; ++q) split_store(Ap[0], Ap[1], Ap[2], Ap[3], la[q], ra[q], ea[q]);
#pragma unroll
    for (int q = 0; q < BCH; ++q) split_store(Bp[0], Bp[1], Bp[2], Bp[3], lb[q], rb[q], eb[q]);
    if (lead) {
#pragma unroll
      for (int q = 0; q < ACH; ++q) sA[ra_row[q]] = ea[q];
#pragma unroll
      for (int q = 0; q < BCH; ++q) sB[rb_row[q]] = eb[q];
    }
    __syncthreads();
    if (kt + 1 < ntiles) load_tile(kt + 1);
    half8 a[TM][4], an[TM][2], b[TN][4];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int at = (wm + 16 * i + li) * PK + 8 * lk;
#pragma unroll
      for (int pl = 0; pl < 4; ++pl) a[i][pl] = *reinterpret_cast<const half8*>(&Ap[pl][at]);
      an[i][0] = negate(a[i][2]);
      an[i][1] = negate(a[i][3]);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int at = (wn + 16 * j + li) * PK + 8 * lk;
#pragma unroll
      for (int pl = 0; pl < 4; ++pl) b[j][pl] = *reinterpret_cast<const half8*>(&Bp[pl][at]);
    }
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      // row scales of this lane's four output rows
      const int4 sa = *reinterpret_cast<const int4*>(&sA[wm + 16 * i + 4 * lk]);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        floatx4 cr = mfma16(a[i][0], b[j][1], zero);      // re: hi*lo + lo*hi + hi*hi
        cr = mfma16(a[i][1], b[j][0], cr);
        cr = mfma16(an[i][0], b[j][3], cr);                // - im * im
        cr = mfma16(an[i][1], b[j][2], cr);
        cr = mfma16(a[i][0], b[j][0], cr);
        cr = mfma16(an[i][0], b[j][2], cr);
        floatx4 ci = mfma16(a[i][0], b[j][3], zero);       // im: re*im + im*re
        ci = mfma16(a[i][1], b[j][2], ci);
        ci = mfma16(a[i][2], b[j][1], ci);
        ci = mfma16(a[i][3], b[j][0], ci);
        ci = mfma16(a[i][0], b[j][2], ci);
        ci = mfma16(a[i][2], b[j][0], ci);
        const int sb = sB[wn + 16 * j + li];
        accr[i][j][0] += ldexpf(cr[0], -(sa.x + sb));
        acci[i][j][0] += ldexpf(ci[0], -(sa.x + sb));
        accr[i][j][1] += ldexpf(cr[1], -(sa.y + sb));
        acci[i][j][1] += ldexpf(ci[1], -(sa.y + sb));
        accr[i][j][2] += ldexpf(cr[2], -(sa.z + sb));
        acci[i][j][2] += ldexpf(ci[2], -(sa.z + sb));
        accr[i][j][3] += ldexpf(cr[3], -(sa.w + sb));
        acci[i][j][3] += ldexpf(ci[3], -(sa.w + sb));
      }
    }
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        int m = wm + 16 * i + 4 * lk + r;
        int n = wn + 16 * j + li;
        if (m0 + m < Mt && n0 + n < Nt) {
          c64 v;
          v.x = accr[i][j][r];
          v.y = acci[i][j][r];
          Out[offCm[m] + offCn[n]] = v;
        }
      }
}

template <int BM, int BN, int WGM>
hipError_t launch_tile_h(const c64* A, const c64* B, c64* Out, const GemmArgs& g, hipStream_t s) {
  dim3 grid((g.M.total + BM - 1) / BM, (g.N.total + BN - 1) / BN, g.L.total);
  hipLaunchKernelGGL((k_gemm_h<BM, BN, WGM>), grid, dim3(256), 0, s, A, B, Out, g);
  return hipGetLastError();
}

template <typename C>
__global__ __launch_bounds__(256) void k_sum_partials(const C* P, C* Out, const Group gm, const Group gn,
                                                      uint32_t mt, uint64_t mn, int parts) {
  const uint64_t o = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (o >= mn) return;
  int32_t pm, cm, pn, cn;
  group_offsets(gm, (uint32_t)(o % mt), pm, cm);
  group_offsets(gn, (uint32_t)(o / mt), pn, cn);
  double re = 0.0, im = 0.0;
  for (int z = 0; z < parts; ++z) {
    const C v = P[(uint64_t)z * mn + o];
    re += (double)v.x;
    im += (double)v.y;
  }
  C r;
  r.x = (decltype(r.x))re;
  r.y = (decltype(r.y))im;
  Out[(int64_t)cm + cn] = r;
}

}  // namespace

int gemm_k_limit() { return (int)GEMM_K_MAX; }

template <typename C>
hipError_t launch_sum_partials(const C* P, C* Out, const Group& gm, const Group& gn, uint32_t mt, uint64_t mn,
                               int parts, hipStream_t s) {
  if (mt < 1 || mn < 1 || parts < 1 || mn % mt != 0 || (uint64_t)gm.total != mt || (uint64_t)gn.total != mn / mt)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_sum_partials<C>), dim3((unsigned)((mn + 255) / 256)), dim3(256), 0, s, P, Out, gm, gn, mt,
                     mn, parts);
  return hipGetLastError();
}
template hipError_t launch_sum_partials<c128>(const c128*, c128*, const Group&, const Group&, uint32_t, uint64_t,
                                              int, hipStream_t);
template hipError_t launch_sum_partials<c64>(const c64*, c64*, const Group&, const Group&, uint32_t, uint64_t, int,
                                             hipStream_t);

template <typename C>
hipError_t launch_gemm(const C* A, const C* B, C* Out, const GemmArgs& g, hipStream_t s) {
  if (g.K.total > GEMM_K_MAX || g.L.total < 1 || g.L.total > 65535) return hipErrorInvalidValue;
  switch (g.tile) {
    case 0: return launch_tile<C, 32, 32, 2>(A, B, Out, g, s);
    case 1: return launch_tile<C, 64, 32, 2>(A, B, Out, g, s);
    case 2: return launch_tile<C, 32, 64, 2>(A, B, Out, g, s);
    case 3: return launch_tile<C, 64, 64, 2>(A, B, Out, g, s);
    case 4: return launch_tile<C, 128, 64, 2>(A, B, Out, g, s);
    case 5: return launch_tile<C, 64, 128, 2>(A, B, Out, g, s);
    case 6: return launch_tile<C, 64, 16, 4>(A, B, Out, g, s);
    case 7: return launch_tile<C, 128, 16, 4>(A, B, Out, g, s);
    case 8: return launch_tile<C, 256, 16, 4>(A, B, Out, g, s);
    case 9: return launch_tile<C, 16, 64, 1>(A, B, Out, g, s);
    case 10: return launch_tile<C, 128, 32, 4>(A, B, Out, g, s);
    case 11: return launch_tile<C, 128, 128, 2>(A, B, Out, g, s);
    case 12: return launch_tile<C, 16, 128, 1>(A, B, Out, g, s);
    case 13: return launch_tile<C, 16, 256, 1>(A, B, Out, g, s);
    case 14: return launch_tile<C, 32, 128, 1>(A, B, Out, g, s);
    default: return hipErrorInvalidValue;
  }
}

bool gemm16_applicable(const GemmArgs& g) {
  return g.contig && g.K.nmodes > 0 && g.K.m[0].ext.d % 32 == 0 && g.K.total <= GEMM_K_MAX &&
         g.L.total >= 1 && g.L.total <= 65535;
}

hipError_t launch_gemm16(const c64* A, const c64* B, c64* Out, const GemmArgs& g, hipStream_t s) {
  if (!gemm16_applicable(g)) return hipErrorInvalidValue;
  switch (g.tile) {
    case 0: return launch_tile_h<32, 32, 2>(A, B, Out, g, s);
    case 1: return launch_tile_h<64, 32, 2>(A, B, Out, g, s);
    case 2: return launch_tile_h<32, 64, 2>(A, B, Out, g, s);
    case 4: return launch_tile_h<128, 64, 2>(A, B, Out, g, s);
    case 5: return launch_tile_h<64, 128, 2>(A, B, Out, g, s);
    case 6: return launch_tile_h<64, 16, 4>(A, B, Out, g, s);
    case 7: return launch_tile_h<128, 16, 4>(A, B, Out, g, s);
    case 9: return launch_tile_h<16, 64, 1>(A, B, Out, g, s);
    case 10: return launch_tile_h<128, 32, 4>(A, B, Out, g, s);
    case 12: return launch_tile_h<16, 128, 1>(A, B, Out, g, s);
    case 14: return launch_tile_h<32, 128, 1>(A, B, Out, g, s);
    default: return launch_tile_h<64, 64, 2>(A, B, Out, g, s);     // 3, and 8 / 11 / 13 (LDS)
  }
}

template hipError_t launch_gemm<c128>(const c128*, const c128*, c128*, const GemmArgs&, hipStream_t);
template hipError_t launch_gemm<c64>(const c64*, const c64*, c64*, const GemmArgs&, hipStream_t);
