// spmv.hpp -- the inner product of the matrix-vector kernels (solver.hip,
// batch.hip), L lanes per row or per node of three rows.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ifem {

template <typename T, int W>
struct Pack {
  T v[W];
};

// Row sum: entries m < cnt of v times x at columns ci[m].  The entries go out
// in pairs, a sum for each half; U pairs per lane (2 L U entries of a row in a
// round) are requested before the first is used (past the end the last pair once more, its products dropped;
// left to the compiler the loads of x go out between the products, and the
// batch of k_bspmv takes 72 instead of 61 ms).  Rows start at any entry, so
// the pairs are aligned to one entry only.
template <int L, int U, typename ACC, typename VV, typename V>
__device__ inline ACC row_dot(int l, int cnt, const VV* __restrict__ v,
                              const int32_t* __restrict__ ci, const V* __restrict__ x)
{
  constexpr int W = 2;
  ACC s[W] = {};
  const int nv = cnt / W;
  for (int k0 = 0; k0 < nv; k0 += L * U) {
    Pack<VV, W> a[U];
    Pack<int, W> c[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = k0 + u * L + l;
      const int m = (k < nv ? k : nv - 1) * W;
      __builtin_memcpy(&c[u], ci + m, sizeof(c[u]));
      __builtin_memcpy(&a[u], v + m, sizeof(a[u]));
    }
    ACC xv[U][W];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int j = 0; j < W; j++) xv[u][j] = (ACC)x[c[u].v[j]];
    __builtin_amdgcn_sched_barrier(0); // all loads before the first product
#pragma unroll
    for (int u = 0; u < U; u++) {
      const bool in = k0 + u * L + l < nv;
#pragma unroll
      for (int j = 0; j < W; j++) {
        const ACC t = s[j] + (ACC)a[u].v[j] * xv[u][j];
        s[j] = in ? t : s[j];
      }
    }
  }
  const int m = nv * W + l;
  if (m < cnt) s[0] += (ACC)v[m] * (ACC)x[ci[m]];
  return s[0] + s[1];
}

// The three row sums of a node: cnt neighbour nodes ci[k], whose three values
// per row are consecutive (rows 3 cnt apart); U neighbours per lane in a round.
template <int L, int U, typename ACC, typename VV, typename V>
__device__ inline void node_dots(int l, int cnt, const VV* __restrict__ v,
                                 const int32_t* __restrict__ ci, const V* __restrict__ x,
                                 ACC (&s)[3])
{
  s[0] = s[1] = s[2] = 0;
  for (int k0 = 0; k0 < cnt; k0 += L * U) {
    Pack<VV, 3> a[U][3];
    int c[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = k0 + u * L + l;
      const int m = k < cnt ? k : cnt - 1;
      c[u] = ci[m];
#pragma unroll
      for (int r = 0; r < 3; r++)
        __builtin_memcpy(&a[u][r], v + 3 * ((int64_t)r * cnt + m), sizeof(a[u][r]));
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const bool in = k0 + u * L + l < cnt;
      Pack<V, 3> xv;
      __builtin_memcpy(&xv, x + 3 * (int64_t)c[u], sizeof(xv));
#pragma unroll
      for (int r = 0; r < 3; r++) {
        const ACC t = s[r] + (ACC)a[u][r].v[0] * (ACC)xv.v[0] + (ACC)a[u][r].v[1] * (ACC)xv.v[1] +
                      (ACC)a[u][r].v[2] * (ACC)xv.v[2];
        s[r] = in ? t : s[r];
      }
    }
  }
}

// Sum over the L lanes of a group, the same in every lane.
template <int L, typename ACC>
__device__ inline ACC group_sum(ACC s)
{
#pragma unroll
  for (int off = L / 2; off >= 1; off >>= 1) s += __shfl_xor(s, off, L);
  return s;
}

} // namespace ifem
