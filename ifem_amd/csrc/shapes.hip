// shapes.hip -- row shapes of a sparsity pattern: the column offsets
// (column - row) of the rows, one copy per distinct list.  Spline systems
// numbered line by line have few of them (the interior rows of a patch share
// one, rows near its faces clip it), so that a product reads one 4-byte shape
// start per row and a small table that stays in the caches instead of 4 bytes
// per nonzero.
//
// Built on the device: a 64-bit hash of every row's list, radix sort, the
// first row of every run gives the list of its shape; every row is then
// compared with its shape's list entry by entry, and any difference (a hash
// collision) drops the shapes.  Patterns whose lists are mostly distinct
// (fixed DOFs strewn over the patch) keep their column indices: the table must
// be at most an eighth of them.  So do small systems, whose products read the
// indices from the caches as fast (cubes of linear scalar elements, FP64: 28^3
// 4.4 us with shapes, 3.4 without; 40^3 4.9 and 5.1; 90^3 36.6 and 46.6): there
// the search would be up to nine tenths of a pattern's set-up.
#include <hip/hip_runtime.h>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include <cstdint>
#include <string>

#include "internal.hpp"

namespace ifem {

// Rows of the pattern: row r has cols[begin(r)] .. of count(r); nodal: node
// triples (rows 3r, 3r+1, 3r+2 share the list of node columns).
struct ShapeRows {
  const int64_t* rowptr;
  const int32_t* cols;
  int nodal;
  __device__ int64_t begin(int r) const { return nodal ? rowptr[3 * (int64_t)r] / 9 : rowptr[r]; }
  __device__ int count(int r) const
  {
    return nodal ? (int)((rowptr[3 * (int64_t)r + 1] - rowptr[3 * (int64_t)r]) / 3)
                 : (int)(rowptr[r + 1] - rowptr[r]);
  }
};

// Finaliser of the splitmix64 generator (Steele, Lea and Flood, 2014).
__device__ inline uint64_t mix64(uint64_t z)
{
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// One wave per row: sum over its entries of a hash of (position, offset).
__global__ void k_shape_hash(ShapeRows R, int n, uint64_t* __restrict__ key, int* __restrict__ row)
{
  const int lane = threadIdx.x & 63;
  const int nw = (int)((gridDim.x * blockDim.x) >> 6);
  for (int r = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6); r < n; r += nw) {
    const int64_t b = R.begin(r);
    const int cnt = R.count(r);
    uint64_t h = 0;
    for (int k = lane; k < cnt; k += 64)
      h += mix64(((uint64_t)(uint32_t)k << 32) ^ (uint64_t)(uint32_t)(R.cols[b + k] - r));
    for (int off = 32; off >= 1; off >>= 1) h += __shfl_xor(h, off, 64);
    if (lane == 0) {
      key[r] = mix64(h ^ ((uint64_t)cnt << 40));
      row[r] = r;
    }
  }
}

// head[i] = 1 where a new shape starts among the sorted keys, len[i] its length.
__global__ void k_shape_heads(ShapeRows R, int n, const uint64_t* __restrict__ key,
                              const int* __restrict__ row, int* __restrict__ head,
                              int* __restrict__ len)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const bool h = i == 0 || key[i] != key[i - 1];
  head[i] = h;
  len[i] = h ? R.count(row[i]) : 0;
}

// start[row] = table start of the row's shape.
__global__ void k_shape_assign(int n, const int* __restrict__ row, const int64_t* __restrict__ incl,
                               ShapeRows R, int32_t* __restrict__ start)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  // incl[i]: total length of the heads up to i; this shape's list is its last part
  start[row[i]] = (int32_t)(incl[i] - R.count(row[i]));
}

// The list of every shape from its first row (one wave per row).
__global__ void k_shape_table(ShapeRows R, int n, const int* __restrict__ row,
                              const int* __restrict__ head, const int32_t* __restrict__ start,
                              int32_t* __restrict__ table)
{
  const int lane = threadIdx.x & 63;
  const int nw = (int)((gridDim.x * blockDim.x) >> 6);
  for (int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6); i < n; i += nw) {
    if (!head[i]) continue;
    const int r = row[i];
    const int64_t b = R.begin(r);
    const int cnt = R.count(r);
    for (int k = lane; k < cnt; k += 64) table[start[r] + k] = R.cols[b + k] - r;
  }
}

// Every row against its shape.  total bounds the reads: a colliding row with
// another length could point outside the table.
__global__ void k_shape_check(ShapeRows R, int n, int total, const int32_t* __restrict__ start,
                              const int32_t* __restrict__ table, int* __restrict__ bad)
{
  const int lane = threadIdx.x & 63;
  const int nw = (int)((gridDim.x * blockDim.x) >> 6);
  for (int r = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6); r < n; r += nw) {
    const int64_t b = R.begin(r);
    const int cnt = R.count(r), st = start[r];
    if (st < 0 || st + cnt > total) {
      if (lane == 0) *bad = 1;
      continue;
    }
    for (int k = lane; k < cnt; k += 64)
      if (table[st + k] != R.cols[b + k] - r) *bad = 1;
  }
}

__global__ void k_shape_clear(int* bad) { *bad = 0; }

static int build(hipStream_t s, int n, const ShapeRows& R, int64_t entries, RowShapes& out,
                 void* work, size_t work_bytes, void*& tmp)
{
  size_t tb = 0, tb2 = 0;
  IFEM_HIP(rocprim::radix_sort_pairs(nullptr, tb, (uint64_t*)nullptr, (uint64_t*)nullptr, (int*)nullptr,
                                     (int*)nullptr, (size_t)n, 0, 64, s));
  IFEM_HIP(rocprim::inclusive_scan(nullptr, tb2, (int*)nullptr, (int64_t*)nullptr, (size_t)n,
                                   rocprim::plus<int64_t>(), s));
  if (tb2 > tb) tb = tb2;
  // without memory for the search the products keep the column indices
  auto alloc = [](void** p, size_t bytes) {
    if (hipMalloc(p, bytes) == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
  };
  const size_t rows = (size_t)n, head_bytes = 40 * rows + 16, need = (head_bytes + 255) / 256 * 256 + tb;
  if (need > work_bytes) {
    if (!alloc(&tmp, need)) return IFEM_GPU_OK;
    work = tmp;
  }
  uint64_t *key = static_cast<uint64_t*>(work), *skey = key + n;
  int64_t* incl = reinterpret_cast<int64_t*>(skey + n);
  int* bad = reinterpret_cast<int*>(incl + n); // two words
  int *row = bad + 2, *srow = row + n, *head = srow + n, *len = head + n;
  void* sort_tmp = static_cast<char*>(work) + (head_bytes + 255) / 256 * 256;
  const unsigned nb = (unsigned)((n + 255) / 256), nwv = (unsigned)((n + 3) / 4 < 8192 ? (n + 3) / 4 : 8192);
  k_shape_hash<<<nwv, 256, 0, s>>>(R, n, key, row);
  IFEM_HIP(rocprim::radix_sort_pairs(sort_tmp, tb, key, skey, row, srow, (size_t)n, 0, 64, s));
  k_shape_heads<<<nb, 256, 0, s>>>(R, n, skey, srow, head, len);
  IFEM_HIP(rocprim::inclusive_scan(sort_tmp, tb, len, incl, (size_t)n, rocprim::plus<int64_t>(), s));
  int64_t total = 0;
  IFEM_HIP(hipMemcpyAsync(&total, incl + n - 1, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  IFEM_HIP(hipStreamSynchronize(s));
  if (total > entries / 8 || total > INT32_MAX) return IFEM_GPU_OK; // mostly distinct
  // three more: the FP16 product reads the list in fours
  if (!alloc((void**)&out.start, sizeof(int32_t) * (size_t)n) ||
      !alloc((void**)&out.table, sizeof(int32_t) * (size_t)(total + 3))) {
    out.release();
    return IFEM_GPU_OK;
  }
  k_shape_assign<<<nb, 256, 0, s>>>(n, srow, incl, R, out.start);
  k_shape_table<<<nwv, 256, 0, s>>>(R, n, srow, head, out.start, out.table);
  k_shape_clear<<<1, 1, 0, s>>>(bad);
  k_shape_check<<<nwv, 256, 0, s>>>(R, n, (int)total, out.start, out.table, bad);
  IFEM_HIP(hipGetLastError());
  int h = 1;
  IFEM_HIP(hipMemcpyAsync(&h, bad, sizeof(int), hipMemcpyDeviceToHost, s));
  IFEM_HIP(hipStreamSynchronize(s));
  if (h) out.release();
  return IFEM_GPU_OK;
}

// Column indices that the products read from the caches as fast as row shapes:
// 4 MB, an XCD's L2.
constexpr int64_t kMinEntries = 1 << 20;

int build_row_shapes(hipStream_t s, int n, const int64_t* rowptr, const int32_t* cols, bool nodal,
                     int64_t entries, void* work, size_t work_bytes, RowShapes& out)
{
  out.release();
  if (n <= 0 || entries < kMinEntries) return IFEM_GPU_OK;
  void* tmp = nullptr;
  const int rc = build(s, n, ShapeRows{rowptr, cols, nodal ? 1 : 0}, entries, out, work, work_bytes, tmp);
  hipFree(tmp);
  if (rc) out.release();
  return rc;
}

void RowShapes::release()
{
  hipFree(start);
  hipFree(table);
  start = table = nullptr;
}

} // namespace ifem
