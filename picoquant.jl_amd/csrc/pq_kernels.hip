// Bandwidth-bound contraction kernels for gfx950 (64-wide wavefronts).
//
//  k_stream  : big x small pairwise contraction (gate application, absorbing
//              a rank-1 output tensor, outer products with a small factor).
//              One lane owns one X-open index; the small operand Y sits in LDS
//              as a dense [K][N] table, so the big operand is read once and C
//              written once -- the HBM roofline for bond-dimension-2 steps.
//  k_generic : any shape; one lane per output element, loop over K.
//  k_reduce  : tiny output (M*N <= 16) with a long summed extent: split-K
//              partial sums per workgroup, then a deterministic second pass.
//  k_copy    : strided gather into contiguous column-major storage
//              (materialises permuted / sliced views).
#include "pq_internal.h"

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace {

template <typename C>
__device__ __forceinline__ C czero() { C r; r.x = 0; r.y = 0; return r; }

// One element, past the caches when NT (non-temporal).
template <bool NT, typename C>
__device__ __forceinline__ C load_one(const C* p) {
  typedef decltype(C::x) V __attribute__((ext_vector_type(2)));
  if constexpr (!NT) return *p;
  return __builtin_bit_cast(C, __builtin_nontemporal_load(reinterpret_cast<const V*>(p)));
}
template <bool NT, typename C>
__device__ __forceinline__ void store_one(C* p, const C& v) {
  typedef decltype(C::x) V __attribute__((ext_vector_type(2)));
  if constexpr (NT)
    __builtin_nontemporal_store(__builtin_bit_cast(V, v), reinterpret_cast<V*>(p));
  else
    *p = v;
}

// ---------------------------------------------------------------- k_stream
// The lane's first X-open index has its K values loaded before the small
// operand is staged in LDS: those loads depend on nothing the staging writes,
// so the kernel waits for global memory once before the barrier, not twice.
// Bound: HBM, or the 256 MB last-level cache where X and Out fit it (7.6 TB/s
// at 2^24 complex64).  NT: X and Out are together too large for that cache,
// so Out (1) or both (2) pass it, and a lane takes one index instead of up
// to 16 (launch_stream has the rule): 2^25 complex64 from three states in turn
// 117 -> 97 us, 2^26 195 -> 167.
template <typename C, int KP, int NT>
__global__ __launch_bounds__(256) void k_stream(const C* __restrict__ X, const C* __restrict__ Y,
                                                C* __restrict__ Out, StreamArgs a) {
  extern __shared__ unsigned char smem_raw[];
  PQ_TOUCH(a.M, a.K, a.N, a.L);
  const uint32_t Kt = a.K.total, Nt = a.N.total, Mt = a.M.total;
  {
    int64_t ox, oy, oc;
    batch_offsets(a.L, blockIdx.z, ox, oy, oc);
    X += ox;
    Y += oy;
    Out += oc;
  }
  // K offsets in X (uniform)
  int32_t xk[KP];
#pragma unroll
  for (int k = 0; k < KP; ++k) {
    int32_t ox = 0, oy = 0;
    if (k < (int)Kt) group_offsets(a.K, (uint32_t)k, ox, oy);
    xk[k] = ox;
  }
  uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
  C xv[KP];
  int32_t oc = 0;
  if (m < Mt) {
    int32_t ox;
    group_offsets(a.M, m, ox, oc);
#pragma unroll
    for (int k = 0; k < KP; ++k) xv[k] = (k < (int)Kt) ? load_one<NT == 2>(X + ox + xk[k]) : czero<C>();
  }
  C* ys = reinterpret_cast<C*>(smem_raw);                              // [KP][Nt]
  int32_t* cn = reinterpret_cast<int32_t*>(ys + (size_t)KP * Nt);      // [Nt]
  for (uint32_t t = threadIdx.x; t < KP * Nt; t += blockDim.x) {
    uint32_t k = t % KP, n = t / KP;
    C v = czero<C>();
    if (k < Kt) {
      int32_t ox, oyk, oyn, ocn;
      group_offsets(a.K, k, ox, oyk);
      group_offsets(a.N, n, oyn, ocn);
      v = Y[oyk + oyn];
    }
    ys[(size_t)n * KP + k] = v;
  }
  for (uint32_t t = threadIdx.x; t < Nt; t += blockDim.x) {
    int32_t oy, ocn;
    group_offsets(a.N, t, oy, ocn);
    cn[t] = ocn;
  }
  __syncthreads();
  for (bool first = true; m < Mt; m += gridDim.x * blockDim.x, first = false) {
    if (!first) {
      int32_t ox;
      group_offsets(a.M, m, ox, oc);
#pragma unroll
      for (int k = 0; k < KP; ++k) xv[k] = (k < (int)Kt) ? load_one<NT == 2>(X + ox + xk[k]) : czero<C>();
    }
    for (uint32_t n = 0; n < Nt; ++n) {
      C acc = czero<C>();
      const C* yc = ys + (size_t)n * KP;
#pragma unroll
      for (int k = 0; k < KP; ++k) cfma(acc, xv[k], yc[k]);
      store_one<NT != 0>(Out + oc + cn[n], acc);
    }
  }
}

// --------------------------------------------------------------- k_generic
// One output per lane, a serial sum over K: along the run of K's first mode
// the addresses step, and only its start is decoded.
// Bound: the chain of loads (7 x 6 outputs over 2933 complex128 values 124 us,
// 671 with every K value decoded; 13 x 11 over 2^10 in ten modes 400 and 633).
template <typename C>
__global__ __launch_bounds__(256) void k_generic(const C* __restrict__ A, const C* __restrict__ B,
                                                 C* __restrict__ Out, GenArgs a) {
  PQ_TOUCH(a.M, a.N, a.K, a.L);
  const uint32_t Mt = a.M.total, Nt = a.N.total, Kt = a.K.total;
  const uint64_t total = (uint64_t)Mt * Nt;
  {
    int64_t oa, ob, oc;
    batch_offsets(a.L, blockIdx.z, oa, ob, oc);
    A += oa;
    B += ob;
    Out += oc;
  }
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total;
       t += (uint64_t)gridDim.x * blockDim.x) {
    uint32_t m = (uint32_t)(t % Mt), n = (uint32_t)(t / Mt);
    int32_t oa, oc1, ob, oc2;
    group_offsets(a.M, m, oa, oc1);
    group_offsets(a.N, n, ob, oc2);
    C acc = czero<C>();
    if (Kt == 1) {                                  // an outer product
      cfma(acc, A[oa], B[ob]);
      Out[oc1 + oc2] = acc;
      continue;
    }
    const uint32_t run = a.K.m[0].ext.d;
    const int32_t sa = a.K.m[0].s0, sb = a.K.m[0].s1;
    for (uint32_t k = 0; k < Kt; k += run) {
      int32_t ka, kb;
      group_offsets(a.K, k, ka, kb);
      ka += oa;
      kb += ob;
      cfma(acc, A[ka], B[kb]);
#pragma unroll 4
      for (uint32_t r = 1; r < run; ++r) cfma(acc, A[ka += sa], B[kb += sb]);
    }
    Out[oc1 + oc2] = acc;
  }
}

// ---------------------------------------------------------------- k_reduce
// Phase 1: workgroup b sums its K chunk for all outputs at once (at most TM x
// TN of them, padded to powers of two): every K value reads each operand row
// once.  partials[b * MN + o]; with a single workgroup the outputs
// themselves.
// With power-of-two K modes an offset is the sum of its index bits': a lane's
// own 8 bits are decoded once, and the wave's 64 lanes decode the uniform
// parts of its next 64 steps together (decoded per step on the scalar unit,
// 23 modes held the loop at 68 us where the loads alone take 46).
// Bound: HBM for long K (2^23 against 2^23 complex128: 180 us before, 53.5
// now at 53 for the bytes), the launches for short (a call on 2^14 x 2^13
// elements closed over 2^13: 39 us on 2 workgroups, 15 on 16; an overlap of
// two 12-qubit states 14 us in two launches, 11 in one).
template <typename C, int TM, int TN>
__global__ __launch_bounds__(256) void k_reduce_partial(const C* __restrict__ A, const C* __restrict__ B,
                                                        C* __restrict__ partials, C* __restrict__ Out, GenArgs a) {
  __shared__ C red[4][TM * TN];
  PQ_TOUCH(a.K, a.M, a.N, a.L);
  const uint32_t Mt = a.M.total, Nt = a.N.total, Kt = a.K.total;
  const uint32_t MN = Mt * Nt;
  {
    int64_t oa, ob, oc;
    batch_offsets(a.L, blockIdx.z, oa, ob, oc);
    A += oa;
    B += ob;
    Out += oc;
  }
  int32_t om[TM], on[TN];
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    int32_t oc = 0;
    om[m] = 0;
    if (m < (int)Mt) group_offsets(a.M, (uint32_t)m, om[m], oc);
  }
#pragma unroll
  for (int n = 0; n < TN; ++n) {
    int32_t oc = 0;
    on[n] = 0;
    if (n < (int)Nt) group_offsets(a.N, (uint32_t)n, on[n], oc);
  }
  const uint32_t chunk = ((Kt + gridDim.x - 1) / gridDim.x + 255) / 256 * 256;
  const uint32_t k0 = blockIdx.x * chunk;
  const uint32_t k1 = min(Kt, k0 + chunk);
  C acc[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = czero<C>();
  // U values of K at a time, so that their loads are in flight together.
  // Rows past the operands' extents read the first row; their sums are not
  // stored.
  constexpr int U = TM + TN <= 4 ? 4 : (TM + TN <= 8 ? 2 : 1);
  auto add = [&](const int32_t (&ka)[U], const int32_t (&kb)[U], int live) {
    C x[U][TM], y[U][TN];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < live) {
#pragma unroll
        for (int m = 0; m < TM; ++m) x[u][m] = A[om[m] + ka[u]];
#pragma unroll
        for (int n = 0; n < TN; ++n) y[u][n] = B[on[n] + kb[u]];
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < live) {
#pragma unroll
        for (int m = 0; m < TM; ++m)
#pragma unroll
          for (int n = 0; n < TN; ++n) cfma(acc[m][n], x[u][m], y[u][n]);
      }
  };
  if (a.K.pow2 && Kt >= 256) {
    // a wave's lanes decode the uniform parts of 64 steps in one go
    int32_t la, lb;
    group_offsets(a.K, threadIdx.x, la, lb);
    for (uint32_t kb = k0; kb < k1; kb += 256 * 64) {
      const uint32_t mine = kb + 256 * (threadIdx.x & 63);
      int32_t va = 0, vb = 0;
      if (mine < k1) group_offsets(a.K, mine, va, vb);
      const int steps = (int)min(64u, (k1 - kb) / 256);
      for (int i = 0; i < steps; i += U) {
        int32_t ka[U], kq[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int t = min(i + u, steps - 1);
          ka[u] = __builtin_amdgcn_readlane(va, t) + la;
          kq[u] = __builtin_amdgcn_readlane(vb, t) + lb;
        }
        if (i + U <= steps)
          add(ka, kq, U);
        else
          add(ka, kq, steps - i);
      }
    }
  } else {
    for (uint32_t k = k0 + threadIdx.x; k < k1; k += 256 * U) {
      int32_t ka[U], kq[U];
      int live = 0;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        ka[u] = kq[u] = 0;
        if (k + 256 * u < k1) {
          group_offsets(a.K, k + 256 * u, ka[u], kq[u]);
          live = u + 1;
        }
      }
      add(ka, kq, live);
    }
  }
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      for (int w = 32; w > 0; w >>= 1) {
        acc[m][n].x += __shfl_xor(acc[m][n].x, w);
        acc[m][n].y += __shfl_xor(acc[m][n].y, w);
      }
      if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64][m + TM * n] = acc[m][n];
    }
  __syncthreads();
  const int t = (int)threadIdx.x, m = t % TM, n = t / TM;
  if (t < TM * TN && m < (int)Mt && n < (int)Nt) {
    C v = red[0][t];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      v.x += red[w][t].x;
      v.y += red[w][t].y;
    }
    if (gridDim.x == 1) {
      int32_t oa, oc1, ob, oc2;
      group_offsets(a.M, (uint32_t)m, oa, oc1);
      group_offsets(a.N, (uint32_t)n, ob, oc2);
      Out[oc1 + oc2] = v;
    } else {
      partials[((size_t)blockIdx.z * gridDim.x + blockIdx.x) * MN + m + Mt * n] = v;
    }
  }
}

// Phase 2: one workgroup per output sums the partials in a fixed order.
template <typename C>
__global__ __launch_bounds__(256) void k_reduce_final(const C* __restrict__ partials, C* __restrict__ Out,
                                                      GenArgs a, int nblocks) {
  __shared__ C red[256];
  const uint32_t Mt = a.M.total, Nt = a.N.total;
  const uint32_t MN = Mt * Nt;
  const uint32_t o = blockIdx.x;
  {
    int64_t oa, ob, oc;
    batch_offsets(a.L, blockIdx.z, oa, ob, oc);
    Out += oc;
  }
  partials += (size_t)blockIdx.z * nblocks * MN;
  C acc = czero<C>();
  for (int b = threadIdx.x; b < nblocks; b += blockDim.x) {
    C p = partials[(size_t)b * MN + o];
    acc.x += p.x; acc.y += p.y;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      red[threadIdx.x].x += red[threadIdx.x + w].x;
      red[threadIdx.x].y += red[threadIdx.x + w].y;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    uint32_t m = o % Mt, n = o / Mt;
    int32_t oa, oc1, ob, oc2;
    group_offsets(a.M, m, oa, oc1);
    group_offsets(a.N, n, ob, oc2);
    Out[oc1 + oc2] = red[0];
  }
}

// ------------------------------------------------------------------ k_copy
template <typename C>
__global__ __launch_bounds__(256) void k_copy(const C* __restrict__ In, C* __restrict__ Out, CopyArgs a) {
  const uint32_t T = a.G.total;
  for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < T; t += gridDim.x * blockDim.x) {
    int32_t oi, oo;
    group_offsets(a.G, t, oi, oo);
    Out[oo] = In[oi];
  }
}

// -------------------------------------------------------------------- k_put
struct PutWords {
  uint32_t w[PQ_PUT_WORDS];
};
__global__ __launch_bounds__(PQ_PUT_WORDS) void k_put(uint32_t* __restrict__ dst, PutWords a, int n) {
  if ((int)threadIdx.x < n) dst[threadIdx.x] = a.w[threadIdx.x];
}

// ------------------------------------------------------------- k_copy_bits
// One tile per workgroup: loaded along its input runs, put into LDS, stored
// along its output runs.  The offsets are sums over index bits, a lane's
// low 8 bits once, the rest uniform, where k_copy decodes every element
// through all modes and reads one element of each line it touches.
// Bound: HBM (2^24 complex64 elements in a random axis order: 48 us = 5.5
// TB/s, 107 us by k_copy, whose time is its per-element decode).  NT: In and
// Out are together well over the 256 MB last-level cache and Out passes it
// (2^24 complex128 in six random orders: three tensors in turn 103-126 us
// cached, 97-126 past it, one of them slower; one again and again 101-126 and
// 67-76).
template <typename C, bool NT>
__global__ __launch_bounds__(256) void k_copy_bits(const C* __restrict__ In, C* __restrict__ Out, CopyBitsArgs a) {
  constexpr int NB = CB_BITS(sizeof(C)), PER = 1 << (NB - 8);
  __shared__ C tile[1 << NB];
  int32_t bi, bo;
  group_offsets(a.outer, blockIdx.x, bi, bo);
  const int tid = threadIdx.x;
  int32_t li = 0, lo = 0, ai = 0, ao = 0;
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const int32_t m = -((tid >> b) & 1);
    li += m & a.is[b];
    lo += m & a.os[b];
    ai ^= m & a.il[b];
    ao ^= m & a.ol[b];
  }
  const C* in = In + bi;
  C* out = Out + bo;
  C v[PER];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    int32_t o = li;
#pragma unroll
    for (int b = 8; b < NB; ++b)
      if ((q >> (b - 8)) & 1) o += a.is[b];
    v[q] = in[o];
  }
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    int32_t t = ai;
#pragma unroll
    for (int b = 8; b < NB; ++b)
      if ((q >> (b - 8)) & 1) t ^= a.il[b];
    tile[t] = v[q];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    int32_t o = lo, t = ao;
#pragma unroll
    for (int b = 8; b < NB; ++b)
      if ((q >> (b - 8)) & 1) {
        o += a.os[b];
        t ^= a.ol[b];
      }
    store_one<NT>(out + o, tile[t]);
  }
}

// ----------------------------------------------------------------- k_multi
// Grouped small contractions: one lane per output element (strided over the
// problem's workgroups of one batch entry), loop over K; a problem may
// instead be a small element-type conversion.  Every problem has just the
// workgroups it needs, found by comparing with the first one of each: a grid
// of (most workgroups) x problems x (most batch entries) started 40960 of
// them for some 700 with work where a wide and a batched problem met (25 us,
// half a nanosecond for an empty one; 7 us now).  NP: 16 problems at most, or
// 64 (a table for 64 alone cost every launch half a microsecond).
template <int NP>
struct MultiFirst {
  uint32_t at[NP];   // past the last problem: none
};
template <typename C, int NP>
__global__ __launch_bounds__(256) void k_multi(const MultiDesc* __restrict__ descs, MultiFirst<NP> first,
                                               int64_t group) {
  int p = 0;
  uint32_t start = 0;
#pragma unroll
  for (int i = 1; i < NP; ++i) {
    p = blockIdx.x >= first.at[i] ? i : p;
    start = blockIdx.x >= first.at[i] ? first.at[i] : start;
  }
  const MultiDesc& d = descs[p];
  PQ_TOUCH(d.M, d.N, d.K, d.L);
  const uint32_t entry = fdiv_q(blockIdx.x - start, d.blocks);
  const uint32_t block = blockIdx.x - start - entry * d.blocks.d;
  int64_t oa, ob, oc;
  batch_offsets(d.L, entry, oa, ob, oc);
  for (int j = 0; j < d.nhigh; ++j)
    if ((group >> j) & 1) {
      oa += d.hA[j];
      ob += d.hB[j];
      oc += d.hC[j];
    }
  if (d.conv) {
    // element-type conversion (complex128 <-> complex64), same layout
    typedef typename std::conditional<sizeof(C) == 16, c64, c128>::type D;
    const C* A = reinterpret_cast<const C*>(d.A) + oa;
    D* Out = reinterpret_cast<D*>(d.C) + oc;
    for (uint32_t t = block * blockDim.x + threadIdx.x; t < d.M.total; t += d.blocks.d * blockDim.x) {
      const C v = A[t];
      D w;
      w.x = (decltype(w.x))v.x;
      w.y = (decltype(w.y))v.y;
      Out[t] = w;
    }
    return;
  }
  const C* A = reinterpret_cast<const C*>(d.A) + oa;
  const C* B = reinterpret_cast<const C*>(d.B) + ob;
  C* Out = reinterpret_cast<C*>(d.C) + oc;
  const uint32_t Mt = d.M.total, Nt = d.N.total, Kt = d.K.total;
  const uint32_t total = Mt * Nt;
  // the problem's K offsets in LDS (grouped problems have K <= PQ_MULTI_KMAX),
  // so a lane issues the loads of eight K values at once instead of waiting
  // for each before decoding the next
  __shared__ int2 kof[PQ_MULTI_KMAX];
  const bool tab = Kt <= PQ_MULTI_KMAX;
  if (tab) {
    for (uint32_t k = threadIdx.x; k < Kt; k += blockDim.x) {
      int32_t ka, kb;
      group_offsets(d.K, k, ka, kb);
      kof[k] = make_int2(ka, kb);
    }
    __syncthreads();
  }
  for (uint32_t t = block * blockDim.x + threadIdx.x; t < total; t += d.blocks.d * blockDim.x) {
    uint32_t m = t % Mt, n = t / Mt;
    int32_t pa, pc1, pb, pc2;
    group_offsets(d.M, m, pa, pc1);
    group_offsets(d.N, n, pb, pc2);
    C acc = czero<C>();
    uint32_t k = 0;
    if (tab) {
      for (; k + 8 <= Kt; k += 8) {
        C a[8], b[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int2 o = kof[k + u];
          a[u] = A[pa + o.x];
          b[u] = B[pb + o.y];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) cfma(acc, a[u], b[u]);
      }
      for (; k < Kt; ++k) {
        const int2 o = kof[k];
        cfma(acc, A[pa + o.x], B[pb + o.y]);
      }
    } else {
      for (; k < Kt; ++k) {
        int32_t ka, kb;
        group_offsets(d.K, k, ka, kb);
        cfma(acc, A[pa + ka], B[pb + kb]);
      }
    }
    Out[pc1 + pc2] = acc;
  }
}

// ------------------------------------------------------------------ k_forest
// One item: an output element of a small unbatched step (one lane, the K
// offsets from the step's table), or one element of a conversion.
template <typename C>
__device__ __forceinline__ void forest_item(const ForestStep& f, const int4& it, const int2* ktab, char* dat) {
  // an operand in the tree's LDS data area holds its byte offset there
  auto at = [&](const void* q, int bit) -> char* {
    return ((f.lds >> bit) & 1) ? dat + (size_t)q : reinterpret_cast<char*>(const_cast<void*>(q));
  };
  if (f.conv) {
    typedef typename std::conditional<sizeof(C) == 16, c64, c128>::type D;
    const C v = reinterpret_cast<const C*>(at(f.A, 0))[it.y];
    D w;
    w.x = (decltype(w.x))v.x;
    w.y = (decltype(w.y))v.y;
    reinterpret_cast<D*>(at(f.C, 2))[it.w] = w;
    return;
  }
  const C* A = reinterpret_cast<const C*>(at(f.A, 0)) + it.y;
  const C* B = reinterpret_cast<const C*>(at(f.B, 1)) + it.z;
  C acc = czero<C>();
  // the loads of several K values in flight at once (a tree's level waits
  // for its slowest lane)
#pragma unroll 4
  for (int32_t k = 0; k < f.nk; ++k) {
    const int2 o = ktab[k];
    cfma(acc, A[o.x], B[o.y]);
  }
  reinterpret_cast<C*>(at(f.C, 2))[it.w] = acc;
}

// Workgroup b runs tree b level by level: a level's items (the outputs of
// all its steps, which read only earlier levels) are spread over the lanes,
// and the barrier after each level makes its stores visible to the
// workgroup's later levels (one workgroup runs on one CU).  Tree header at
// lv[lv[b]]: levels, first step record, step records, first K entry, K
// entries, first leaf copy, leaf copies, then the levels' item bounds.
// LDS: the tree's step records and K offsets are copied into LDS once, so
// a level waits on global memory only for its operands (the items of the
// next level are read ahead, as they depend on nothing the level computes);
// the results that the tree itself reads later, and the small leaves it
// reads, live in the LDS data area after them (leaves copied in at the
// start), so only the other leaves and the tree's root result go through
// global memory.
// Bound: the levels' latency, one after another.  1024 lanes, since a level
// of a few thousand outputs left 256 with several in turn: 24 us instead of
// 38 for 44 trees of 16 levels, 33 instead of 44 for 69 (512 lanes: a
// microsecond longer).
template <bool LDS>
__global__ __launch_bounds__(PQ_FOREST_LANES) void k_forest(const ForestStep* __restrict__ fs, const int4* __restrict__ items,
                                                const int2* __restrict__ ktab,
                                                const ForestCopy* __restrict__ copies,
                                                const int32_t* __restrict__ lv) {
  extern __shared__ __align__(16) int32_t fsm[];
  const int32_t q = lv[blockIdx.x];
  const int32_t nlev = lv[q], fs0 = lv[q + 1], nfs = lv[q + 2], k0 = lv[q + 3], nkt = lv[q + 4];
  const int32_t c0 = lv[q + 5], nc = lv[q + 6];
  const int32_t* bnd = lv + q + 7;
  const ForestStep* F = fs + fs0;
  const int2* KT = ktab + k0;
  char* dat = nullptr;
  if constexpr (LDS) {
    constexpr int W = (int)(sizeof(ForestStep) / 4);
    const int tid = (int)threadIdx.x;
    // leaf copies first: their loads are in flight while the records move
    float2 cv[PQ_FOREST_COPY_PER_LANE];
    int32_t cd[PQ_FOREST_COPY_PER_LANE];
#pragma unroll
    for (int j = 0; j < PQ_FOREST_COPY_PER_LANE; ++j) {
      const int32_t e = tid + PQ_FOREST_LANES * j;
      if (e < nc) {
        const ForestCopy cp = copies[c0 + e];
        cv[j] = *reinterpret_cast<const float2*>(cp.src);
        cd[j] = cp.dst;
      }
    }
    const int32_t* src = reinterpret_cast<const int32_t*>(fs + fs0);
    for (int32_t e = tid; e < nfs * W; e += (int32_t)blockDim.x) fsm[e] = src[e];
    const int32_t kw = nfs * W + (nfs * W & 1);
    int2* kd = reinterpret_cast<int2*>(fsm + kw);
    for (int32_t e = tid; e < nkt; e += (int32_t)blockDim.x) kd[e] = ktab[k0 + e];
    dat = reinterpret_cast<char*>(fsm) + (((size_t)kw * 4 + (size_t)nkt * 8 + 15) & ~(size_t)15);
#pragma unroll
    for (int j = 0; j < PQ_FOREST_COPY_PER_LANE; ++j)
      if (tid + PQ_FOREST_LANES * j < nc) *reinterpret_cast<float2*>(dat + cd[j]) = cv[j];
    __syncthreads();
    F = reinterpret_cast<const ForestStep*>(fsm);
    KT = kd;
  }
  int4 nx = make_int4(0, 0, 0, 0);
  if (nlev > 0 && bnd[0] + (int32_t)threadIdx.x < bnd[1]) nx = items[bnd[0] + threadIdx.x];
  for (int32_t l = 0; l < nlev; ++l) {
    const int32_t i0 = bnd[l] + (int32_t)threadIdx.x, i1 = bnd[l + 1];
    const int4 cur = nx;
    if (l + 1 < nlev && i1 + (int32_t)threadIdx.x < bnd[l + 2]) nx = items[i1 + threadIdx.x];
    // the lane's next items of this level, loaded together (a level of a
    // few thousand outputs gives a lane several)
    constexpr int PRE = 3;
    int4 pre[PRE];
#pragma unroll
    for (int j = 0; j < PRE; ++j) {
      const int32_t i = i0 + (j + 1) * (int32_t)blockDim.x;
      if (i < i1) pre[j] = items[i];
    }
    int32_t c = 0;
    for (int32_t i = i0; i < i1; i += (int32_t)blockDim.x, ++c) {
      int4 it;
      if (c == 0) {
        it = cur;
      } else if (c <= PRE) {
        it = pre[0];
        if (c == 2) it = pre[1];
        if (c == 3) it = pre[2];
      } else {
        it = items[i];
      }
      const ForestStep& f = F[it.x - fs0];
      if (f.c128)
        forest_item<c128>(f, it, KT + (f.kt - k0), dat);
      else
        forest_item<c64>(f, it, KT + (f.kt - k0), dat);
    }
    __syncthreads();
  }
}

inline unsigned grid_for(uint64_t work, unsigned block, unsigned cap = 8192) {
  uint64_t g = (work + block - 1) / block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (unsigned)g;
}

}  // namespace

template <typename C>
hipError_t launch_stream(const C* X, const C* Y, C* Out, const StreamArgs& a, hipStream_t s) {
  const uint32_t Kt = a.K.total, Nt = a.N.total;
  int KP = 1;
  while ((uint32_t)KP < Kt) KP <<= 1;
  size_t smem = (size_t)KP * Nt * sizeof(C) + (size_t)Nt * 4;
  // X and Out together well over the last level's 256 MB pass the caches,
  // Out or both, and a lane takes one index (or 64 bytes of X and Out), on up
  // to 65536 workgroups.  Measured a gate at a time, each on the last one's
  // result, us cached / Out passing / both passing, by the position of the
  // bits summed:
  //   complex64, 512 MB:  4 and 5 99 / 93 / 90, 1 and 9 99 / 92 / 95, 0 and 1
  //     102 / 91 / 119, 0 to 2 110 / 107 / 183; 2 GB: 435 / 371 / 364, 433 /
  //     369 / 389, 434 / 369 / 494, 442 / 404 / 733
  //   complex128, 1 GB:  0 206 / 189 / 184, 1 and 9 206 / 209 / 200, 0 and 1
  //     209 / 188 / 280, 5 to 7 206 / 219 / 203; 5 and 8 onto one 150 / 141 /
  //     133; 512 MB: 0 97 / 97 / 93, 1 and 9 101 / 108 / 103, 0 and 1 105 / 96
  //     / 143, 5 to 7 101 / 114 / 109
  // so X passes only where its first mode runs over a whole 128-byte line (a
  // shorter run is read by several loads, each fetching the line anew) or with
  // two K values of 16 bytes.  complex128 stays cached from four K values on,
  // unless Out is narrow or a lane's K values lie together; one index a lane
  // still pays for four K values and 1 GB (1 and 9 206 -> 198, 2 GB 437 ->
  // 397; eight K values 206 -> 213, 512 MB 101 -> 100 and up to 115).
  // 256 MB together: 35-43 us cached, 47-54 passing.  Where the caches serve,
  // more than 4096 workgroups are an eighth slower (each stages Y).
  const double mb = (double)a.M.total * a.L.total * (Kt + Nt) * sizeof(C) / (1 << 20);
  const bool line = a.M.nmodes > 0 && a.M.m[0].s0 == 1 && (uint64_t)a.M.m[0].ext.d * sizeof(C) >= 128;
  const bool near = a.K.nmodes == 1 && a.K.m[0].s0 == 1;
  int nt = 0;
  if (mb > 384 && sizeof(C) == 8) nt = line ? 2 : 1;
  if (mb > 384 && sizeof(C) == 16) nt = Kt <= 2 || (Nt <= 2 && line) ? 2 : (near ? 1 : 0);
  const bool wide = nt != 0 || (mb > 640 && sizeof(C) == 16 && Kt <= 4 && Nt <= 4);
  const uint64_t lanes = wide ? a.M.total / std::max<uint64_t>(64 / ((Kt + Nt) * sizeof(C)), 1) : a.M.total;
  const dim3 grid(grid_for(lanes, 256, a.L.total > 1 ? 1024 : (wide ? 65536 : 4096)), 1, a.L.total), block(256);
  switch (KP * 4 + nt) {
#define PQ_CASE2(P, NT) \
  case P * 4 + NT: hipLaunchKernelGGL((k_stream<C, P, NT>), grid, block, smem, s, X, Y, Out, a); break;
#define PQ_CASE(P) PQ_CASE2(P, 0) PQ_CASE2(P, 1) PQ_CASE2(P, 2)
    PQ_CASE(1) PQ_CASE(2) PQ_CASE(4) PQ_CASE(8) PQ_CASE(16) PQ_CASE(32)
#undef PQ_CASE
#undef PQ_CASE2
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename C>
hipError_t launch_generic(const C* A, const C* B, C* Out, const GenArgs& a, hipStream_t s) {
  uint64_t work = (uint64_t)a.M.total * a.N.total;
  hipLaunchKernelGGL((k_generic<C>), dim3(grid_for(work, 256, a.L.total > 1 ? 1024 : 8192), 1, a.L.total),
                     dim3(256), 0, s, A, B, Out, a);
  return hipGetLastError();
}

int reduce_blocks_for(uint32_t ktotal, uint32_t batch, uint32_t outputs) {
  // one workgroup, which needs no second launch, for up to 4096 values of K
  // and 2^15 products (2 x 2 outputs over 4096: 6.3 us, 9.6 in eight parts;
  // 16 over 2048 12.3 and 13.2, over 4096 16.2 and 13.1)
  if (ktotal <= 4096 && (uint64_t)ktotal * outputs <= 1u << 15) return 1;
  // 4096 values per workgroup (16 per lane) and at most 2048 workgroups;
  // fewer values, down to 512, while that keeps the device short of 2048
  const uint32_t least = ktotal / 4096, fill = std::min(ktotal / 512, 2048u / std::max(batch, 1u));
  return (int)std::min(std::max(std::max(least, fill), 1u), 2048u);
}

template <typename C, int TM, int TN>
static void reduce_partial(const C* A, const C* B, C* Out, const GenArgs& a, C* partials, int nblocks, hipStream_t s) {
  hipLaunchKernelGGL((k_reduce_partial<C, TM, TN>), dim3(nblocks, 1, a.L.total), dim3(256), 0, s, A, B, partials, Out,
                     a);
}

template <typename C>
hipError_t launch_reduce(const C* A, const C* B, C* Out, const GenArgs& a, C* partials, int nblocks,
                         hipStream_t s) {
  auto log2up = [](uint32_t v) {
    int l = 0;
    while ((1u << l) < v) ++l;
    return l;
  };
  const int lm = log2up(a.M.total), ln = log2up(a.N.total);
  switch (lm * 8 + ln) {
#define PQ_CASE(LM, LN) \
  case LM * 8 + LN: reduce_partial<C, 1 << LM, 1 << LN>(A, B, Out, a, partials, nblocks, s); break;
    PQ_CASE(0, 0) PQ_CASE(0, 1) PQ_CASE(0, 2) PQ_CASE(0, 3) PQ_CASE(0, 4) PQ_CASE(1, 0) PQ_CASE(1, 1) PQ_CASE(1, 2)
    PQ_CASE(1, 3) PQ_CASE(2, 0) PQ_CASE(2, 1) PQ_CASE(2, 2) PQ_CASE(2, 3) PQ_CASE(3, 0) PQ_CASE(3, 1) PQ_CASE(3, 2)
    PQ_CASE(4, 0)
#undef PQ_CASE
    default: return hipErrorInvalidValue;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || nblocks == 1) return e;
  hipLaunchKernelGGL((k_reduce_final<C>), dim3(a.M.total * a.N.total, 1, a.L.total), dim3(256), 0, s, partials,
                     Out, a, nblocks);
  return hipGetLastError();
}

template <typename C>
hipError_t launch_copy(const C* In, C* Out, const CopyArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((k_copy<C>), dim3(grid_for(a.G.total, 256)), dim3(256), 0, s, In, Out, a);
  return hipGetLastError();
}

hipError_t launch_put(void* dst, const void* host, int n, hipStream_t s) {
  if (n < 1 || n > PQ_PUT_WORDS) return hipErrorInvalidValue;
  PutWords a;
  memcpy(a.w, host, (size_t)n * 4);
  hipLaunchKernelGGL(k_put, dim3(1), dim3(n <= 64 ? 64 : PQ_PUT_WORDS), 0, s, (uint32_t*)dst, a, n);
  return hipGetLastError();
}

template <typename C>
hipError_t launch_copy_bits(const C* In, C* Out, const CopyBitsArgs& a, hipStream_t s) {
  const dim3 grid(a.outer.total), block(256);
  if (2.0 * a.outer.total * (1 << CB_BITS(sizeof(C))) * sizeof(C) > 384.0 * (1 << 20))
    hipLaunchKernelGGL((k_copy_bits<C, true>), grid, block, 0, s, In, Out, a);
  else
    hipLaunchKernelGGL((k_copy_bits<C, false>), grid, block, 0, s, In, Out, a);
  return hipGetLastError();
}

template <typename C, int NP>
static void launch_problems(const MultiDesc* descs, const uint32_t* wgs, int n, int64_t group, hipStream_t s) {
  MultiFirst<NP> first;
  uint32_t total = 0;
  for (int i = 0; i < NP; ++i) {
    first.at[i] = i < n ? total : UINT32_MAX;
    if (i < n) total += wgs[i];
  }
  hipLaunchKernelGGL((k_multi<C, NP>), dim3(total), dim3(256), 0, s, descs, first, group);
}

template <typename C>
hipError_t launch_multi(const MultiDesc* descs, const std::vector<uint32_t>& wgs, int64_t group, hipStream_t s) {
  for (size_t p = 0; p < wgs.size(); p += 64) {
    const int n = (int)std::min<size_t>(wgs.size() - p, 64);
    if (n <= 16)
      launch_problems<C, 16>(descs + p, wgs.data() + p, n, group, s);
    else
      launch_problems<C, 64>(descs + p, wgs.data() + p, n, group, s);
  }
  return hipGetLastError();
}

hipError_t launch_forest(const ForestStep* steps, const int4* items, const int2* ktab, const ForestCopy* copies,
                         const int32_t* lv, int ntrees, size_t lds_bytes, hipStream_t s) {
  if (ntrees < 1 || ntrees > (1 << 24) || lds_bytes > PQ_FOREST_LDS_BYTES) return hipErrorInvalidValue;
  if (lds_bytes > 0)
    hipLaunchKernelGGL(k_forest<true>, dim3(ntrees), dim3(PQ_FOREST_LANES), lds_bytes, s, steps, items, ktab, copies, lv);
  else
    hipLaunchKernelGGL(k_forest<false>, dim3(ntrees), dim3(PQ_FOREST_LANES), 0, s, steps, items, ktab, copies, lv);
  return hipGetLastError();
}

#define PQ_INST(C)                                                                                   \
  template hipError_t launch_multi<C>(const MultiDesc*, const std::vector<uint32_t>&, int64_t, hipStream_t); \
  template hipError_t launch_stream<C>(const C*, const C*, C*, const StreamArgs&, hipStream_t);      \
  template hipError_t launch_generic<C>(const C*, const C*, C*, const GenArgs&, hipStream_t);        \
  template hipError_t launch_reduce<C>(const C*, const C*, C*, const GenArgs&, C*, int, hipStream_t); \
  template hipError_t launch_copy<C>(const C*, C*, const CopyArgs&, hipStream_t);                    \
  template hipError_t launch_copy_bits<C>(const C*, C*, const CopyBitsArgs&, hipStream_t);
PQ_INST(c128)
PQ_INST(c64)
