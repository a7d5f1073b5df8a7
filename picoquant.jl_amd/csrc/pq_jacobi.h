// Small truncated SVD split on the GPU (pq_jacobi.hip).
#pragma once
#include "pq_common.h"

#include <algorithm>
#include <cstddef>
#include <vector>

#define JAC_MAX_Q 64        // shorter side
#define JAC_MAX_SWEEPS 30

struct JacMeta {
  double root[JAC_MAX_Q];   // sqrt of column c's singular value
  double rest[JAC_MAX_Q];   // ... and what its rounding left
  int32_t pos[JAC_MAX_Q];   // its place in descending order
  int32_t chi, lines;
};

struct JacArgs {
  const void* X;            // m x n through gm (rows, s0) and gn (columns, s0)
  Group gm, gn;
  int32_t m, n, p, q, trans;   // p, q, trans: filled by launch_jacobi
  void* Q;                  // scratch, max(m, n) x min(m, n)
  void* log;                // scratch, jacobi_log_bytes
  JacMeta* meta;            // scratch
  void *B, *C;              // m x chi and chi x n, room for min(m, n) (max_rank if given) of chi
  double thr;               // cut-off relative to the spectrum's 2-norm
  int32_t max_rank;
  int32_t* host;            // pinned: chi, 1 if the sweeps did not converge
};

// Whether an m x n matrix of elements of es bytes runs on it.
bool jacobi_fits(int64_t m, int64_t n, size_t es);
size_t jacobi_log_bytes(int64_t q, size_t es);
template <typename C>
hipError_t launch_jacobi(JacArgs j, hipStream_t s);
