// Whether the rows of a KV cache, as its strides describe them, are memory of their own.
#pragma once
#include <cstdint>

#include "../../include/mimir_prefixlm.h"

namespace mimir {

struct LayoutDim {
  int64_t n, stride;
};

// Whether every index of the dims has an address of its own: true if, by ascending
// stride, each stride reaches past all that the smaller ones span (every layout that
// slices, permutes or interleaves a dense one; expanded and overlapping ones fail, and
// so may an unusual distinct one).
inline bool distinct_addresses(LayoutDim* dims, int count) {
  for (int i = 1; i < count; ++i)
    for (int j = i; j > 0 && dims[j].stride < dims[j - 1].stride; --j) {
      const LayoutDim t = dims[j];
      dims[j] = dims[j - 1];
      dims[j - 1] = t;
    }
  int64_t span = 1;
  for (int i = 0; i < count; ++i) {
    if (dims[i].n <= 1) continue;
    if (dims[i].stride < span) return false;
    span += (dims[i].n - 1) * dims[i].stride;
  }
  return true;
}

// Whether no two (tensor, cache row, position, kv head) rows of the call's two cache
// tensors share memory, among the cache rows that the call can reach.  Expanded caches
// (a batch stride of 0: every batch row on the same positions), overlapping windows and
// one tensor for keys and values do.
inline bool cache_rows_distinct(const MimirCacheAttnParams& p) {
  const int64_t rows = p.batch_indices != nullptr || p.cache_rows < p.batch ? p.cache_rows : p.batch;
  if (rows <= 0 || p.cache_len <= 0) return true;
  LayoutDim k[5] = {{rows, p.ck_stride_batch}, {p.cache_len, p.ck_stride_token}, {p.num_kv_heads, p.ck_stride_head},
                    {p.head_dim, 1}, {1, 0}};
  LayoutDim v[4] = {{rows, p.cv_stride_batch}, {p.cache_len, p.cv_stride_token}, {p.num_kv_heads, p.cv_stride_head},
                    {p.head_dim, 1}};
  const uintptr_t a = (uintptr_t)p.cache_k, b = (uintptr_t)p.cache_v;  // bf16: 2 bytes an element
  uintptr_t ka = a, vb = b;  // one past the last byte
  for (int i = 0; i < 4; ++i) {
    ka += 2 * (uintptr_t)((k[i].n - 1) * k[i].stride);
    vb += 2 * (uintptr_t)((v[i].n - 1) * v[i].stride);
  }
  ka += 2;
  vb += 2;
  if (ka <= b || vb <= a) return distinct_addresses(k, 4) && distinct_addresses(v, 4);
  // Interleaved: keys and values as one more dim of a single layout.
  for (int i = 0; i < 3; ++i)
    if (k[i].n > 1 && k[i].stride != v[i].stride) return false;
  k[4] = {2, (int64_t)((a < b ? b - a : a - b) / 2)};
  return distinct_addresses(k, 5);
}

}  // namespace mimir
