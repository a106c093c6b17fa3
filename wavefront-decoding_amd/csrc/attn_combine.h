// What the attention kernels that split long prefixes share: the split width,
// the merge of a row's split partials, the partials' workspace, and the row
// tables of a packed varlen call.
#pragma once

#include "wfd_common.h"

namespace wfd {

constexpr int kAttnSplit = 1024;  // keys per workgroup

__device__ __forceinline__ float attn_finish(float O, float L) { return L > 0.f ? O / L : 0.f; }

// Merge of a row's split partials, in split order: M = max m_s, then
// L = sum l_s * 2^(m_s - M) and O = sum o_s * 2^(m_s - M), one fma per split.
// The partials are read in batches of kCombineBatch independent loads, so a
// row of many splits waits on memory twice per batch, not twice per split.
constexpr int kCombineBatch = 8;

template <typename T, int DH>
__global__ __launch_bounds__(DH) void attn_combine_kernel(const float* __restrict__ part_o,
                                                          const float* __restrict__ part_ml,
                                                          const int32_t* __restrict__ kv_len, T* __restrict__ out,
                                                          int H, int max_splits) {
  constexpr int B = kCombineBatch;
  const int h = blockIdx.x;
  const int i = blockIdx.y;
  const int d = threadIdx.x;
  const int len = kv_len[i];
  int ns = len > 0 ? (len + kAttnSplit - 1) / kAttnSplit : 0;
  ns = min(ns, max_splits);
  if (ns <= 1) return;  // finished by its split workgroup
  const int64_t base = ((int64_t)i * H + h) * max_splits;
  float M = -INFINITY;
  for (int s0 = 0; s0 < ns; s0 += B) {
    float mv[B];
#pragma unroll
    for (int b = 0; b < B; ++b) mv[b] = s0 + b < ns ? part_ml[(base + s0 + b) * 2] : -INFINITY;
#pragma unroll
    for (int b = 0; b < B; ++b) M = fmaxf(M, mv[b]);
  }
  float O = 0.f, L = 0.f;
  for (int s0 = 0; s0 < ns; s0 += B) {
    float mv[B], lv[B], ov[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const bool ok = s0 + b < ns;
      mv[b] = ok ? part_ml[(base + s0 + b) * 2] : -INFINITY;
      lv[b] = ok ? part_ml[(base + s0 + b) * 2 + 1] : 0.f;
      ov[b] = ok ? part_o[(base + s0 + b) * DH + d] : 0.f;
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
      if (s0 + b < ns) {
        const float f = (mv[b] == -INFINITY) ? 0.f : exp2f(mv[b] - M);
        L = fmaf(lv[b], f, L);
        O = fmaf(ov[b], f, O);
      }
    }
  }
  Elem<T>::store(out + ((int64_t)i * H + h) * DH + d, attn_finish(O, L));
}

// Row r of a packed varlen call (the FA varlen convention): query row r of
// segment s (rows [cu_q[s], cu_q[s+1]), keys [cu_k[s], cu_k[s+1]) of a
// token-major K / V) reads keys from row cu_k[s]; non-causal it reads the
// whole segment, causal (bottom-right) keys [0, k_len - q_len + r - cu_q[s]].
// Rows before cu_q[0] or at or past cu_q[nseg] get no keys. A binary search
// over cu_q: the tables never leave the device.
__device__ __forceinline__ void varlen_row(const int32_t* __restrict__ cu_q, const int32_t* __restrict__ cu_k,
                                           int nseg, int causal, int r, int64_t& row_base, int32_t& kv_len) {
  int lo = 0, hi = nseg;  // find the last s with cu_q[s] <= r
  if (nseg <= 0 || r >= cu_q[nseg] || r < cu_q[0]) {
    row_base = 0;
    kv_len = 0;
    return;
  }
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cu_q[mid] <= r)
      lo = mid;
    else
      hi = mid;
  }
  const int qs = cu_q[lo], ql = cu_q[lo + 1] - qs;
  const int ks = cu_k[lo], kl = cu_k[lo + 1] - ks;
  row_base = ks;
  kv_len = causal ? max(kl - ql + (r - qs) + 1, 0) : kl;
}

inline int max_splits_for(int kv_len_max) { return kv_len_max <= 0 ? 1 : (kv_len_max + kAttnSplit - 1) / kAttnSplit; }

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

inline size_t attn_ws_bytes(int n, int H, int Dh, int kv_len_max) {
  const size_t ms = (size_t)max_splits_for(kv_len_max);
  return align256((size_t)n * H * ms * Dh * sizeof(float)) + align256((size_t)n * H * ms * 2 * sizeof(float));
}

}  // namespace wfd
