// Packed varlen attention for segments of several query rows (bf16), on MFMA.
//
// Replaces: fa4_attention.attn_varlen / _attn_varlen_torch
//   (src/decoding/fa4_attention.py:301-317,348-366) where a segment brings more
//   than one row: chunked prompts, a coda's verifies, re-entered tokens.
//
// Same operation as the row form (varlen row tables + wfd_attn_decode): query
// row r of a segment attends the segment's first kv_len[r] keys; softmax and
// sums in fp32. The row form streams a row's whole prefix once per row; here a
// workgroup owns a tile of 32 / G rows of one segment (G = H / Hkv query heads
// per kv head: 32 (row, head) pairs, one per lane column of a 32x32 MFMA) and
// one kv head, and reads each key once for all of them.
//
// What bounds it: with up to 32 rows per key the call is a stream of K and V
// (at 48 segments of 1-64 rows over 100-2048 keys x 16 heads x 128: 394 MB),
// so the layout keeps loads in flight: 4 waves take the 32-key tiles of a
// 1024-key split round-robin, each with its own LDS block and no barrier in the
// loop; a tile's 16 KB are loaded into registers (whole key rows, 1 KB per
// instruction) while the tile before it is computed. Two workgroups per CU fit
// by LDS (80 KB each at Dh 128, Q's fragments among them: in registers they made
// the loop spill), so one streams while the other merges. That shape takes 124
// us (the tables 5, this kernel 111, the merge of splits 10; 3.5 TB/s) against
// 720 us for the row form; what is left is the ragged last round of 1540
// workgroups over 512 places. Two S^T chains instead of one changed nothing.
//
// Arithmetic: S^T = K Q^T and O^T = V^T P^T on v_mfma_f32_32x32x16_bf16, V^T
// read from the row-major tile with the transposing LDS read, keys permuted
// inside a tile so that the S^T accumulators are the P^T operand in place
// (lane half hf, register rr: key 16 (rr / 8) + 8 hf + rr % 8). The
// probabilities enter the second product as two bf16 terms, p = hi + lo (16
// significant bits), each its own MFMA into the same fp32 sum, so they are not
// rounded to bf16: the output's error against float64 is that of the row form
// (1.7e-3, the bf16 output rounding; with hi alone 2.0e-3). A row's bits depend
// on its own keys only, not on its tile, its column or the other segments: key
// tiles go to waves and splits by key index, masked keys add exact zeros.
// Waves merge through LDS in wave order, splits in split order
// (attn_combine_kernel).
#include "attn_combine.h"

namespace wfd {

constexpr int kRowsCols = 32;   // (row, head) pairs per workgroup
constexpr int kRowsWaves = 4;
constexpr int kRowsKeys = 32;   // keys per tile

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 rows_mfma(const u32x4& a, const u32x4& b, f32x16 acc) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc,
                                                 0, 0, 0);
}

// Tiles of at most `qt` rows, none across a segment boundary: tile i holds rows
// [first[i], first[i + 1]), entries past the last tile repeat total_q (empty
// tiles). The rows before cu_q[0] and from cu_q[nseg] on (no keys) are tiled
// too: their output rows are zeros. One workgroup.
__device__ __forceinline__ void varlen_tiles(const int32_t* __restrict__ cu_q, int nseg, int total_q, int qt,
                                             int32_t* __restrict__ first, int cap) {
  __shared__ int scan[256];
  __shared__ int base;
  const int tid = threadIdx.x;
  if (tid == 0) base = 0;
  auto start = [&](int s) {  // first row of part s: 0, the segments, the rows past them
    if (s <= 0) return 0;
    if (s > nseg + 1) return total_q;
    return min(max(cu_q[s - 1], 0), total_q);
  };
  __syncthreads();
  for (int s0 = 0; s0 < nseg + 2; s0 += 256) {
    const int s = s0 + tid;
    const int a = s < nseg + 2 ? start(s) : 0;
    const int b = s < nseg + 2 ? start(s + 1) : 0;
    const int count = b > a ? (b - a + qt - 1) / qt : 0;
    scan[tid] = count;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
      const int v = tid >= d ? scan[tid - d] : 0;
      __syncthreads();
      scan[tid] += v;
      __syncthreads();
    }
    const int off = base + scan[tid] - count;
    for (int i = 0; i < count; ++i)
      if (off + i < cap) first[off + i] = a + i * qt;
    const int sum = scan[255];
    __syncthreads();  // every thread has read base and the scan
    if (tid == 0) base += sum;
    __syncthreads();
  }
  for (int i = base + tid; i < cap; i += 256) first[i] = total_q;
}

// Row tables (all workgroups but the last) and the tile table (the last).
__global__ __launch_bounds__(256) void varlen_tables_kernel(const int32_t* __restrict__ cu_q,
                                                            const int32_t* __restrict__ cu_k, int nseg, int total_q,
                                                            int causal, int qt, int64_t* __restrict__ row_base,
                                                            int32_t* __restrict__ kv_len,
                                                            int32_t* __restrict__ tile_first, int cap) {
  if (blockIdx.x + 1 == gridDim.x) {
    varlen_tiles(cu_q, nseg, total_q, qt, tile_first, cap);
    return;
  }
  const int r = blockIdx.x * 256 + threadIdx.x;
  if (r < total_q) varlen_row(cu_q, cu_k, nseg, causal, r, row_base[r], kv_len[r]);
}

// Grid (Hkv x tiles, splits), 256 threads.
template <int DH, int G>
__global__ __launch_bounds__(64 * kRowsWaves) __attribute__((amdgpu_waves_per_eu(2))) void attn_rows_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
    const int64_t* __restrict__ row_base, const int32_t* __restrict__ kv_len, const int32_t* __restrict__ tile_first,
    float* __restrict__ part_o, float* __restrict__ part_ml, bf16_t* __restrict__ out, int H, int Hkv, int max_splits,
    float scale_log2) {
  constexpr int V = 8;
  constexpr int NW = kRowsWaves;
  constexpr int QT = kRowsCols / G;        // rows per tile
  constexpr int NDS = DH / 16;             // MFMA k-steps over Dh
  constexpr int NDB = DH / 32;             // 32-row blocks of O^T
  constexpr int VRP = DH + 32;             // padded LDS row of V (elements): spreads a transposing read over all banks
  constexpr int CPR = DH / V;              // 16-byte pieces of a key row
  constexpr int NCH = kRowsKeys * CPR / 64;  // K (and V) pieces per lane per tile
  constexpr int PW = NDB * 16 + 2;         // floats a lane parks for the merge
  constexpr int kWaveLds = kRowsKeys * (DH + VRP) * (int)sizeof(bf16_t);
  static_assert(NW * kWaveLds >= NW * PW * 64 * (int)sizeof(float), "park area");
  static_assert(NDS % NW == 0, "Q fragments staged by wave");
  static_assert(NDB <= NW && kRowsCols % G == 0, "merge split");
  static_assert(kRowsKeys * DH * sizeof(bf16_t) >= kRowsKeys * 32 * sizeof(float), "P in the K tile's LDS");
  __shared__ __align__(16) unsigned char lds[NW * kWaveLds];
  __shared__ __align__(16) u32x4 q_lds[NDS][64];  // Q fragments: 32 registers a lane fewer, or the loop spills

  const int g = blockIdx.x % Hkv;
  const int tile = blockIdx.x / Hkv;
  const int split = blockIdx.y;
  const int r0 = tile_first[tile];
  const int nr = min(tile_first[tile + 1] - r0, QT);
  if (nr <= 0) return;  // empty tile (uniform)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int col = lane & 31;  // this lane's (row, head) pair
  const int hf = lane >> 5;
  const bool real = col / G < nr;
  const int row = r0 + (real ? col / G : 0);
  const int head = g * G + col % G;
  const int lim = real ? max(kv_len[row], 0) : 0;  // keys [0, lim)
  int maxlen = lim, minlen = real ? lim : 0x7fffffff;
#pragma unroll
  for (int m = 16; m >= 1; m >>= 1) {
    maxlen = max(maxlen, __shfl_xor(maxlen, m, 64));
    minlen = min(minlen, __shfl_xor(minlen, m, 64));
  }
  maxlen = __builtin_amdgcn_readfirstlane(maxlen);
  minlen = __builtin_amdgcn_readfirstlane(minlen);
  const int kbeg = split * kAttnSplit;
  if (split > 0 && kbeg >= maxlen) return;  // uniform over the workgroup
  const int nkeys = max(min(maxlen, kbeg + kAttnSplit) - kbeg, 0);  // of this split
  const int nt = (nkeys + kRowsKeys - 1) / kRowsKeys;

  // K / V of this kv head from key kbeg; the resources end at the split's last
  // key, so loads of later keys read zeros and send nothing to memory
  const uint32_t rsb = (uint32_t)(Hkv * DH * sizeof(bf16_t));  // key stride, bytes
  const int64_t hb = ((row_base[r0] + kbeg) * Hkv + g) * DH;
  const uint32_t span = nkeys > 0 ? (uint32_t)(nkeys - 1) * rsb + DH * (uint32_t)sizeof(bf16_t) : 0u;
  const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(kc + hb), (short)0, span,
                                                                      0x00020000);
  const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(vc + hb), (short)0, span,
                                                                      0x00020000);
  bf16_t* const kl = reinterpret_cast<bf16_t*>(lds + wave * kWaveLds);
  bf16_t* const vl = kl + kRowsKeys * DH;
  // K rows unpadded, 16-byte pieces XORed by the row: 16 rows' reads of one piece
  // (and a row's 16 stores) touch every bank once
  auto k_at = [](int key, int piece) {
    return (key * CPR + (piece ^ (CPR == 16 ? key & 15 : (key >> 1) & (CPR - 1)))) * V;
  };

  // Q as the MFMA B operand: column col, dims 16 k + 8 hf + (0..7)
  {
    const bf16_t* qp = q + ((int64_t)row * H + head) * DH + hf * V;
#pragma unroll
    for (int i = 0; i < NDS / NW; ++i) {
      const int k = wave * (NDS / NW) + i;
      q_lds[k][lane] = ld16(qp + k * 16);
    }
  }
  // key (within a tile) of MFMA row col: the permutation above
  const int krow = 16 * ((col >> 3) >> 1) + 8 * ((col >> 2) & 1) + 4 * ((col >> 3) & 1) + (col & 3);

  u32x4 kreg[NCH], vreg[NCH];
  const uint32_t lane_off = (uint32_t)(lane / CPR) * rsb + (uint32_t)(lane % CPR) * 16u;
  auto fetch = [&](int t) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const uint32_t off = lane_off + (uint32_t)(t * kRowsKeys + i * (64 / CPR)) * rsb;
      kreg[i] = buf_ld16(kr, off);
      vreg[i] = buf_ld16(vr, off);
    }
  };
  // V^T fragment of d-block db, key step k (see the prefill kernel): two
  // transposing reads of 4 keys x 16 columns per 16-lane group
  const int tg = lane >> 4, ti = lane & 15;
  const int v_lane = ((tg >> 1) * 8 + (ti >> 2)) * VRP + 16 * (tg & 1) + 4 * (ti & 3);
  auto vt_frag = [&](int db, int k) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    typedef const __attribute__((address_space(3))) void* lds_ptr;
    const bf16_t* p = vl + v_lane + 16 * k * VRP + 32 * db;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(lds_ptr)p);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(lds_ptr)(p + 4 * VRP));
    const uint2 a = __builtin_bit_cast(uint2, lo), c = __builtin_bit_cast(uint2, hi);
    return u32x4{a.x, a.y, c.x, c.y};
  };

  float mrun = -INFINITY, lrun = 0.f;
  f32x16 o[NDB];
#pragma unroll
  for (int c = 0; c < NDB; ++c)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[c][r] = 0.f;

  // Whether a V value of the lane's loaded tile is infinite or NaN. Such a tile
  // leaves the matrix product (0 x infinity for a masked key or a zero low term
  // would reach rows that the value does not belong to) and is added key by key.
  auto v_special = [&]() {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    u16x2 m = {0, 0};
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, vreg[i][e] & 0x7f807f80u));
    return m.x == 0x7f80 || m.y == 0x7f80;
  };

  fetch(wave);
  __syncthreads();  // q_lds
  for (int t = wave; t < nt; t += NW) {  // uniform over the wave; no barrier in the loop
    // the LDS executes one wave's accesses in order: the previous tile's
    // reads, these stores, this tile's reads
    const bool special = __builtin_amdgcn_ballot_w64(v_special()) != 0;  // uniform
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = lane + 64 * i;
      *reinterpret_cast<u32x4*>(kl + k_at(c / CPR, c % CPR)) = kreg[i];
      *reinterpret_cast<u32x4*>(vl + (c / CPR) * VRP + (c % CPR) * V) = vreg[i];
    }
    asm volatile("" ::: "memory");
    fetch(t + NW);  // past the last tile: zeros, no traffic
    f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
    for (int k = 0; k < NDS; ++k)
      s = rows_mfma(*reinterpret_cast<const u32x4*>(kl + k_at(krow, 2 * k + hf)), q_lds[k][lane], s);
    const int k0 = kbeg + t * kRowsKeys;
    if (k0 + kRowsKeys > minlen) {  // some row's last key lies in or before this tile (uniform)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (k0 + 16 * (r >> 3) + 8 * hf + (r & 7) >= lim) s[r] = -INFINITY;
    }
    float mt = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mt = fmaxf(mt, s[r]);
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    const float mnew = fmaxf(mrun, mt * scale_log2);
    const float mref = mnew == -INFINITY ? 0.f : mnew;  // a row with no key so far: every p is 0
    const float corr = __builtin_amdgcn_exp2f(mrun - mref);
    float ls = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], scale_log2, -mref));
      ls += s[r];
    }
    ls += __shfl_xor(ls, 32, 64);
    lrun = fmaf(lrun, corr, ls);
    mrun = mnew;
    if (__builtin_amdgcn_ballot_w64(corr != 1.f)) {
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= corr;
    }
    if (special) {
      // P through the K tile's LDS (its reads are done), one key at a time, then
      // zeros in V's place for the products below
      float* const pl32 = reinterpret_cast<float*>(kl);
      asm volatile("" ::: "memory");
#pragma unroll
      for (int r = 0; r < 16; ++r) pl32[(16 * (r >> 3) + 8 * hf + (r & 7)) * 32 + col] = s[r];
      asm volatile("" ::: "memory");
      for (int key = 0; key < kRowsKeys && k0 + key < maxlen; ++key) {
        const bool mine = k0 + key < lim;
        const float p = mine ? pl32[key * 32 + col] : 0.f;
#pragma unroll
        for (int i = 0; i < 4 * NDB; ++i) {
          const uint2 w = *reinterpret_cast<const uint2*>(vl + key * VRP + 8 * i + 4 * hf);
          f32x16& oo = o[i >> 2];
          const int b = 4 * (i & 3);
          oo[b + 0] = fmaf(p, mine ? bf16_bits_to_f32(w.x & 0xffffu) : 0.f, oo[b + 0]);
          oo[b + 1] = fmaf(p, mine ? bf16_bits_to_f32(w.x >> 16) : 0.f, oo[b + 1]);
          oo[b + 2] = fmaf(p, mine ? bf16_bits_to_f32(w.y & 0xffffu) : 0.f, oo[b + 2]);
          oo[b + 3] = fmaf(p, mine ? bf16_bits_to_f32(w.y >> 16) : 0.f, oo[b + 3]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int c = lane + 64 * i;
        *reinterpret_cast<u32x4*>(vl + (c / CPR) * VRP + (c % CPR) * V) = zero16();
      }
      asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      // p = hi + lo, both bf16: P^T operand of key step k from registers 8k .. 8k + 7
      u32x4 ph, pl;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p0 = s[8 * k + 2 * e], p1 = s[8 * k + 2 * e + 1];
        ph[e] = f32x2_to_bf16x2_bits(p0, p1);
        pl[e] = f32x2_to_bf16x2_bits(p0 - __uint_as_float(ph[e] << 16), p1 - __uint_as_float(ph[e] & 0xffff0000u));
      }
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        const u32x4 vt = vt_frag(db, k);
        o[db] = rows_mfma(vt, ph, o[db]);
        o[db] = rows_mfma(vt, pl, o[db]);
      }
    }
  }

  // merge the waves in wave order: each parks its state (its own LDS block may
  // be another wave's park area: barrier first), then wave db merges d-block db
  __syncthreads();
  float* const park = reinterpret_cast<float*>(lds);
  {
    float* p = park + wave * PW * 64 + lane;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) p[(16 * db + r) * 64] = o[db][r];
    p[16 * NDB * 64] = mrun;
    p[(16 * NDB + 1) * 64] = lrun;
  }
  __syncthreads();
  if (wave >= NDB) return;  // after the last barrier
  const int db = wave;
  float M = -INFINITY, L = 0.f, O[16];
#pragma unroll
  for (int w = 0; w < NW; ++w) M = fmaxf(M, park[(w * PW + 16 * NDB) * 64 + lane]);
#pragma unroll
  for (int r = 0; r < 16; ++r) O[r] = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float* p = park + w * PW * 64 + lane;
    const float mw = p[16 * NDB * 64];
    const float f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);
    L = fmaf(p[(16 * NDB + 1) * 64], f, L);
#pragma unroll
    for (int r = 0; r < 16; ++r) O[r] = fmaf(p[(16 * db + r) * 64], f, O[r]);
  }
  if (!real) return;
  // register r: output column d = 32 db + 8 (r / 4) + 4 hf + r % 4
  const int ns = min((lim + kAttnSplit - 1) / kAttnSplit, max_splits);
  const int64_t oh = (int64_t)row * H + head;
  if (ns <= 1) {
    if (split > 0) return;
    const float inv = L > 0.f ? 1.f / L : 0.f;  // a row without keys: zeros
    bf16_t* op = out + oh * DH + 32 * db + 4 * hf;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint2 w;
      w.x = f32x2_to_bf16x2_bits(O[4 * i] * inv, O[4 * i + 1] * inv);
      w.y = f32x2_to_bf16x2_bits(O[4 * i + 2] * inv, O[4 * i + 3] * inv);
      *reinterpret_cast<uint2*>(op + 8 * i) = w;
    }
  } else if (kbeg < lim) {
    const int64_t pidx = oh * max_splits + split;
    float* op = part_o + pidx * DH + 32 * db + 4 * hf;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<f32x4*>(op + 8 * i) = f32x4{O[4 * i], O[4 * i + 1], O[4 * i + 2], O[4 * i + 3]};
    if (db == 0 && hf == 0) {
      part_ml[pidx * 2] = M;
      part_ml[pidx * 2 + 1] = L;
    }
  }
}

// Workspace of a varlen call: row tables, tile table, split partials.
struct VarlenWs {
  size_t kv_len, tiles, part, bytes;
  int cap;  // tile table entries (tiles + 1)
};

static VarlenWs varlen_ws(int nseg, int total_q, int H, int Hkv, int Dh, int max_k) {
  VarlenWs w{};
  const int qt = kRowsCols / (H / Hkv);
  w.cap = total_q / qt + nseg + 3;
  w.kv_len = align256((size_t)total_q * sizeof(int64_t));
  w.tiles = w.kv_len + align256((size_t)total_q * sizeof(int32_t));
  w.part = w.tiles + align256((size_t)w.cap * sizeof(int32_t));
  w.bytes = w.part + (max_splits_for(max_k) > 1 ? attn_ws_bytes(total_q, H, Dh, max_k) : 0);
  return w;
}

template <int DH, int G>
static void launch_rows(const void* q, const void* k, const void* v, const int64_t* rb, const int32_t* kl,
                        const int32_t* tf, int tiles, float* po, float* pml, void* out, int n, int H, int Hkv, int ms,
                        float scale_log2, hipStream_t st) {
  hipLaunchKernelGGL((attn_rows_kernel<DH, G>), dim3((unsigned)tiles * Hkv, ms), dim3(64 * kRowsWaves), 0, st,
                     (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, rb, kl, tf, po, pml, (bf16_t*)out, H, Hkv,
                     ms, scale_log2);
  if (ms > 1)
    hipLaunchKernelGGL((attn_combine_kernel<bf16_t, DH>), dim3(H, n), dim3(DH), 0, st, po, pml, kl, (bf16_t*)out, H,
                       ms);
}

}  // namespace wfd

extern "C" {

size_t wfd_attn_varlen_workspace_bytes(int nseg, int total_q, int H, int Hkv, int Dh, int max_k) {
  if (nseg < 0 || total_q < 0 || H <= 0 || Hkv <= 0 || H % Hkv != 0 || H / Hkv > wfd::kRowsCols || Dh <= 0) return 0;
  return wfd::varlen_ws(nseg, total_q, H, Hkv, Dh, max_k).bytes;
}

int wfd_attn_varlen(const void* q, const void* k, const void* v, const int32_t* cu_q, const int32_t* cu_k, void* out,
                    int nseg, int total_q, int H, int Hkv, int Dh, int dtype, float scale, int max_k, int causal,
                    void* workspace, size_t ws_bytes, hipStream_t stream) {
  using namespace wfd;
  if (nseg < 0 || total_q < 0 || H <= 0 || Hkv <= 0 || H % Hkv != 0 || max_k < 1) {
    set_error("wfd_attn_varlen: bad shape nseg=%d total_q=%d H=%d Hkv=%d max_k=%d", nseg, total_q, H, Hkv, max_k);
    return kBadArg;
  }
  const int G = H / Hkv;
  if (!(scale > 0.f)) {
    set_error("wfd_attn_varlen: scale=%g must be positive", (double)scale);
    return kBadArg;
  }
  if (dtype != kBF16 || (Dh != 64 && Dh != 128) || (G != 1 && G != 2 && G != 4)) {
    set_error("wfd_attn_varlen: unsupported dtype=%d Dh=%d G=%d (bf16, Dh 64/128, G 1/2/4)", dtype, Dh, G);
    return kUnsupported;
  }
  if (total_q == 0) return kOk;
  if (!q || !k || !v || !cu_q || !cu_k || !out || !workspace) {
    set_error("wfd_attn_varlen: null pointer argument");
    return kBadArg;
  }
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out | (uintptr_t)workspace) & 15) {
    set_error("wfd_attn_varlen: q, k, v, out and workspace must be 16-byte aligned");
    return kBadArg;
  }
  const VarlenWs w = varlen_ws(nseg, total_q, H, Hkv, Dh, max_k);
  if (ws_bytes < w.bytes) {
    set_error("wfd_attn_varlen: workspace %zu bytes < required %zu", ws_bytes, w.bytes);
    return kWorkspace;
  }
  char* base = (char*)workspace;
  int64_t* rb = (int64_t*)base;
  int32_t* kl = (int32_t*)(base + w.kv_len);
  int32_t* tf = (int32_t*)(base + w.tiles);
  const int ms = max_splits_for(max_k);
  float* po = (float*)(base + w.part);
  float* pml = (float*)(base + w.part + align256((size_t)total_q * H * ms * Dh * sizeof(float)));
  hipLaunchKernelGGL(varlen_tables_kernel, dim3((total_q + 255) / 256 + 1), dim3(256), 0, stream, cu_q, cu_k, nseg,
                     total_q, causal ? 1 : 0, kRowsCols / G, rb, kl, tf, w.cap);
  const float sl2 = scale * 1.4426950408889634f;
#define WFD_ROWS_CASE(DHV, GV)                                                                              \
  if (Dh == DHV && G == GV)                                                                                 \
    launch_rows<DHV, GV>(q, k, v, rb, kl, tf, w.cap - 1, po, pml, out, total_q, H, Hkv, ms, sl2, stream);
  WFD_ROWS_CASE(64, 1)
  WFD_ROWS_CASE(64, 2)
  WFD_ROWS_CASE(64, 4)
  WFD_ROWS_CASE(128, 1)
  WFD_ROWS_CASE(128, 2)
  WFD_ROWS_CASE(128, 4)
#undef WFD_ROWS_CASE
  return launch_status("wfd_attn_varlen");
}

}  // extern "C"
