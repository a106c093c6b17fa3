// Packed varlen attention for segments of several query rows (bf16), on MFMA,
// with the decode kernel's bits.
//
// Replaces: fa4_attention.attn_varlen / _attn_varlen_torch
//   (src/decoding/fa4_attention.py:301-317,348-366) where a segment brings more
//   than one row: chunked prompts, a coda's verifies, re-entered tokens.
//
// Same operation as the row form (varlen row tables + wfd_attn_decode): query
// row r of a segment attends the segment's first kv_len[r] keys. The row form
// streams a row's whole prefix once per row; here a workgroup owns a tile of
// 16 / G rows of one segment (G = H / Hkv query heads per kv head: 16 (row, head)
// pairs, one per lane column) and one kv head, and reads each key once for all.
//
// Arithmetic: exactly attn_split_kernel's, value for value, so a row has the
// same bits whichever kernel a call takes and whichever rows ride along:
//  * scores on the same 16x16x32 bf16 product in the same k order, formed
//    transposed (K as the A operand), which leaves a lane with scores of one
//    (row, head) pair: its softmax state is one register each;
//  * the same tile per wave (tile t of a 1024-key split belongs to wave t % 8),
//    and a tile's sum of probabilities in the row form's order: over 16-key
//    blocks, then the xor 8, 4, 2, 1 butterfly over the key within the block;
//  * P.V in fp32 on v_mfma_f32_16x16x4_f32, which is the chain
//    fma(a3,b3,fma(a2,b2,fma(a1,b1,fma(a0,b0,c)))) bit for bit, denormals,
//    infinities and NaN included (checked on the device against fmaf over 7
//    distributions x 10^6 sums: no difference, every other order differs). The
//    row form's lane vg adds keys RG k + vg, k = 0, 1, ..; here that chain is
//    an accumulator of its own, four keys per product (lane group = k), and the
//    keys of a tile are permuted so that a lane's probabilities are the
//    product's B operand in place;
//  * the chains' and the waves' merge in the same order, splits in split order
//    (attn_combine_kernel).
//
// What bounds it: issue. A tile of 16 pairs x 32 keys x 128 columns is 64 fp32
// products of 32 cycles, 44 % of the time that a CU is busy with 48 segments of
// 1-64 rows over 100-2048 keys x 16 heads x 128 (394 MB of K and V), and vector
// instructions another 37 %; the two do not overlap, also across waves. 164 us (the
// tables 5, this kernel 147, the merge of splits 10) against 720 for the row form;
// a fifth of the time CUs wait for the last workgroups. The chains take 128
// registers, so a CU holds 8 waves: as two workgroups of 4 waves with two parts each,
// so that one's loads and merge run under the other's products (one workgroup of 8
// waves: 209 us; with the merge's factors computed once per output 182; with one
// conversion between two products, which costs the matrix core some ten cycles,
// masks and denormal handling in every tile 168). K and V of the next tile are
// loaded as soon as the registers of this one's are free.
#include "attn_combine.h"

namespace wfd {

constexpr int kRowsCols = 16;   // (row, head) pairs per workgroup
constexpr int kRowsParts = 8;   // attn_split_kernel's waves: part w sums tiles w, w + 8, ..
constexpr int kRowsWaves = 4;   // each takes parts w and w + 4 in turn

// (x of the lane with bit 5 / bit 4 of its number clear, x of the one with it set), the
// other bits the lane's own: a butterfly step's two terms without the LDS
struct Pair {
  float a, b;
};
__device__ __forceinline__ Pair pair32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ Pair pair16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return {__uint_as_float(r[0]), __uint_as_float(r[1])};
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
  constexpr int NW = kRowsWaves;
  constexpr int NP = kRowsParts;
  constexpr int QT = kRowsCols / G;   // rows per tile
  constexpr int TK = DH == 64 ? 64 : 32;  // keys per tile, as attn_split_kernel
  constexpr int RG = 512 / DH;        // P.V chains (attn_split_kernel's V row groups)
  constexpr int NJ = TK / 16;         // 16-key blocks of S^T
  constexpr int NDS = DH / 32;        // MFMA k-steps over Dh
  constexpr int NB = DH / 16;         // 16-column blocks of O^T: block b holds columns NB i + b
  constexpr int NS = TK / (4 * RG);   // products per chain and tile
  constexpr int PW = NB / 2;          // 32-bit words of a lane's V piece
  constexpr int OP = DH + 4;          // padded row of the merge area
  static_assert(NJ * 4 == NS * RG && NS == 2, "score registers are the P.V operands");
  __shared__ __align__(16) float o_lds[NP][kRowsCols][OP];
  __shared__ float m_lds[NP][kRowsCols];
  __shared__ float l_lds[NP][kRowsCols];

  const int g = blockIdx.x % Hkv;
  const int tile = blockIdx.x / Hkv;
  const int split = blockIdx.y;
  const int r0 = tile_first[tile];
  const int nr = min(tile_first[tile + 1] - r0, QT);
  if (nr <= 0) return;  // empty tile (uniform)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int col = lane & 15;  // this lane's (row, head) pair; as an A row: its key or column group
  const int grp = lane >> 4;
  const bool real = col / G < nr;
  const int lim = real ? max(kv_len[r0 + col / G], 0) : 0;  // keys [0, lim)
  int maxlen = lim, minlen = real ? lim : 0x7fffffff;
#pragma unroll
  for (int m = 8; m >= 1; m >>= 1) {
    maxlen = max(maxlen, __shfl_xor(maxlen, m, 64));
    minlen = min(minlen, __shfl_xor(minlen, m, 64));
  }
  maxlen = __builtin_amdgcn_readfirstlane(maxlen);
  minlen = __builtin_amdgcn_readfirstlane(minlen);
  const int kbeg = split * kAttnSplit;
  if (split > 0 && kbeg >= maxlen) return;  // uniform over the workgroup
  const int nkeys = max(min(maxlen, kbeg + kAttnSplit) - kbeg, 0);  // of this split
  const int nt = (nkeys + TK - 1) / TK;
  const int np = min(nt, NP);  // parts that hold keys

  // K / V of this kv head from key kbeg; the resources end at the split's last
  // key, so loads of later keys read zeros and send nothing to memory
  const uint32_t rsb = (uint32_t)(Hkv * DH * sizeof(bf16_t));  // key stride, bytes
  const int64_t hb = ((row_base[r0] + kbeg) * Hkv + g) * DH;
  const uint32_t span = nkeys > 0 ? (uint32_t)(nkeys - 1) * rsb + DH * (uint32_t)sizeof(bf16_t) : 0u;
  const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(kc + hb), (short)0, span,
                                                                      0x00020000);
  const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(vc + hb), (short)0, span,
                                                                      0x00020000);

  // Score block j, MFMA row i = 4 grp + r is key RG (4 s + grp) + vg of the tile
  // for the product (s, vg) = (4 j + r) / RG, (4 j + r) % RG: the row form's
  // chain vg at its step k = 4 s + grp
  auto key_of = [](int j, int i) {
    return RG * (4 * (4 * j / RG) + (i >> 2)) + (4 * j) % RG + (i & 3);
  };

  u32x4 kreg[NJ][NDS];
  uint32_t vreg[NS * RG][PW];
  const uint32_t k_lane = (uint32_t)key_of(0, col) * rsb + (uint32_t)grp * 16u;
  const uint32_t v_lane = (uint32_t)(RG * grp) * rsb + (uint32_t)(col * NB * 2);
  auto fetch_k = [&](int t) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const uint32_t off = k_lane + (uint32_t)(t * TK + key_of(j, 0)) * rsb;
#pragma unroll
      for (int s = 0; s < NDS; ++s) kreg[j][s] = buf_ld16(kr, off + s * 64);
    }
  };
  auto fetch_v = [&](int t, int x) {  // piece x = (s, vg): NB columns of key RG (4 s + grp) + vg
    const uint32_t off = v_lane + (uint32_t)(t * TK + 4 * RG * (x / RG) + x % RG) * rsb;
    if constexpr (PW == 4) {
      const u32x4 w = buf_ld16(vr, off);
#pragma unroll
      for (int e = 0; e < 4; ++e) vreg[x][e] = w[e];
    } else {
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      const u32x2 w = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(vr, off, 0, 0));
      vreg[x][0] = w[0];
      vreg[x][1] = w[1];
    }
  };

  auto lo_special = [](uint32_t w) { return (w & 0x7f80u) == 0x7f80u; };  // infinite or NaN
  auto hi_special = [](uint32_t w) { return (w & 0x7f800000u) == 0x7f800000u; };

  fetch_k(wave);
  // Q as the B operand: column col, dims 32 s + 8 grp + (0..7)
  u32x4 qf[NDS];
  {
    const bf16_t* qp = q + ((int64_t)(r0 + (real ? col / G : 0)) * H + g * G + col % G) * DH + grp * 8;
#pragma unroll
    for (int s = 0; s < NDS; ++s) qf[s] = real ? ld16(qp + s * 32) : zero16();
  }
#pragma unroll
  for (int x = 0; x < NS * RG; ++x) fetch_v(wave, x);
#pragma unroll 1
  for (int part = wave; part < np; part += NW) {
    float mrun = -INFINITY, lrun = 0.f;
    f32x4 o[RG][NB];  // O^T by chain: columns NB (4 grp + r) + b of pair col
#pragma unroll
    for (int c = 0; c < RG; ++c)
#pragma unroll
      for (int b = 0; b < NB; ++b) o[c][b] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int t = part; t < nt; t += NP) {  // uniform over the wave; no barrier in the loop
      const int tn = t + NP < nt || part >= NW ? t + NP : part + NW;  // the next tile: of this part, or the wave's other one
      const int t0 = kbeg + t * TK;
      f32x4 p[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        p[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NDS; ++s) p[j] = mfma_step<bf16_t>(kreg[j][s], qf[s], p[j]);
      }
      fetch_k(tn);  // past the last tile: zeros, no traffic
      {
#pragma clang fp contract(off)
        float mt = -INFINITY;
        if (t0 + TK > minlen) {  // some row's last key lies in or before this tile (uniform)
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              p[j][r] = t0 + key_of(j, 4 * grp) + r < lim ? p[j][r] * scale_log2 : -INFINITY;
              mt = fmaxf(mt, p[j][r]);
            }
        } else {
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              p[j][r] *= scale_log2;
              mt = fmaxf(mt, p[j][r]);
            }
        }
        const Pair m32 = pair32(mt);
        const Pair m16 = pair16(fmaxf(m32.a, m32.b));
        mt = fmaxf(m16.a, m16.b);
        const float mnew = fmaxf(mrun, mt);
        const float corr = (mrun == -INFINITY) ? 0.f : exp2f(mrun - mnew);
        mrun = mnew;
        // exp2f(x) is v_exp_f32(x) from -126 up, which is what most tiles hold
        float low = 0.f;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) low = fminf(low, p[j][r] - mnew);
        if (__builtin_amdgcn_ballot_w64(low >= -126.f) == ~0ull) {
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) p[j][r] = __builtin_amdgcn_exp2f(p[j][r] - mnew);
        } else {
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) p[j][r] = (p[j][r] == -INFINITY) ? 0.f : exp2f(p[j][r] - mnew);
        }
        // the tile's sum, by key % 16 (c) over the tile's 16-key blocks, then the
        // butterfly over c: xor 8, 4, 2, 1
        float u[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if constexpr (RG == 4) {  // c = 4 grp + r
            const Pair v = pair32(p[0][r] + p[1][r]);
            const Pair w = pair16(v.a + v.b);
            u[r] = w.a + w.b;
          } else {  // c = 8 (grp & 1) + 4 h + r, 16-key block 2 s + grp / 2
            float w[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const Pair s0 = pair32(p[h][r]), s1 = pair32(p[2 + h][r]);
              const Pair v = pair16(((s0.a + s0.b) + s1.a) + s1.b);
              w[h] = v.a + v.b;
            }
            u[r] = w[0] + w[1];
          }
        }
        lrun = fmaf(lrun, corr, (u[0] + u[2]) + (u[1] + u[3]));
        if (t != part && __builtin_amdgcn_ballot_w64(corr != 1.f)) {  // the first tile: o is 0
#pragma unroll
          for (int c = 0; c < RG; ++c)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
              for (int r = 0; r < 4; ++r) o[c][b][r] *= corr;
        }
      }
      // A tile in which some row's last key lies (uniform): 0 x infinity would
      // reach rows that an infinite or NaN V value does not belong to. Such a value
      // becomes 0 in the products and is added here to the pairs that attend it (to
      // chain 0: which chain holds an infinity or a NaN changes nothing)
      if (t0 + TK > minlen) {
#pragma unroll
        for (int x = 0; x < NS * RG; ++x) {
          bool special = false;
#pragma unroll
          for (int e = 0; e < PW; ++e) special |= lo_special(vreg[x][e]) || hi_special(vreg[x][e]);
          if (__builtin_amdgcn_ballot_w64(special) == 0) continue;
#pragma unroll 1
          for (int k = 0; k < 4; ++k) {  // key RG (4 s + k) + vg: held by lane group k
            const float pk = __shfl(p[x / 4][x % 4], 16 * k + col, 64);
            const bool mine = t0 + RG * (4 * (x / RG) + k) + x % RG < lim;
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
              for (int e = 0; e < PW; ++e) {
                const uint32_t w = __shfl(vreg[x][e], 16 * k + 4 * grp + r, 64);
                if (mine && lo_special(w)) o[0][2 * e][r] = fmaf(pk, __uint_as_float(w << 16), o[0][2 * e][r]);
                if (mine && hi_special(w)) o[0][2 * e + 1][r] = fmaf(pk, __uint_as_float(w & 0xffff0000u), o[0][2 * e + 1][r]);
                __builtin_amdgcn_sched_barrier(0);
              }
          }
#pragma unroll
          for (int e = 0; e < PW; ++e) {
            if (lo_special(vreg[x][e])) vreg[x][e] &= 0xffff0000u;
            if (hi_special(vreg[x][e])) vreg[x][e] &= 0xffffu;
          }
        }
      }
      // eight values converted, then their products: a VALU instruction between two
      // products costs the matrix core some ten cycles
      constexpr int XB = 8 / NB;
#pragma unroll
      for (int x0 = 0; x0 < NS * RG; x0 += XB) {
        float v[XB][NB];
#pragma unroll
        for (int x = 0; x < XB; ++x)
#pragma unroll
          for (int e = 0; e < PW; ++e) {
            v[x][2 * e] = __uint_as_float(vreg[x0 + x][e] << 16);
            v[x][2 * e + 1] = __uint_as_float(vreg[x0 + x][e] & 0xffff0000u);
          }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = x0; x < x0 + XB; ++x)
#pragma unroll
          for (int b = 0; b < NB; ++b)
            o[x % RG][b] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(v[x - x0][b], p[x / 4][x % 4], o[x % RG][b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = x0; x < x0 + XB; ++x) fetch_v(tn, x);
      }
    }

    // the chains in the row form's shuffle order, then the part leaves its state
#pragma unroll
    for (int c = 1; c < RG; c <<= 1)
#pragma unroll
      for (int a = 0; a < RG; a += 2 * c)
#pragma unroll
        for (int b = 0; b < NB; ++b) o[a][b] += o[a + c][b];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int b = 0; b < NB; b += 4)
        *reinterpret_cast<f32x4*>(&o_lds[part][col][NB * (4 * grp + r) + b]) =
            f32x4{o[0][b][r], o[0][b + 1][r], o[0][b + 2][r], o[0][b + 3][r]};
    if (grp == 0) {
      m_lds[part][col] = mrun;
      l_lds[part][col] = lrun;
    }
  }
  __syncthreads();

  // merge and finish as attn_split_kernel, NB columns of one pair per thread
  static_assert(16 * kRowsCols == 64 * NW, "16 threads per pair");
  const int m = threadIdx.x >> 4;
  const int d = (threadIdx.x & 15) * NB;
  if (m >= nr * G) return;
  const int i = r0 + m / G;
  const int64_t oh = (int64_t)i * H + g * G + m % G;
  const int len = kv_len[i];
  float O[NB];
#pragma unroll
  for (int e = 0; e < NB; ++e) O[e] = 0.f;
  auto store = [&](const float (&v)[NB]) {
    uint32_t w[PW];
#pragma unroll
    for (int e = 0; e < PW; ++e) w[e] = f32x2_to_bf16x2_bits(v[2 * e], v[2 * e + 1]);
    if constexpr (PW == 4)
      *reinterpret_cast<u32x4*>(out + oh * DH + d) = u32x4{w[0], w[1], w[2], w[3]};
    else
      *reinterpret_cast<uint2*>(out + oh * DH + d) = uint2{w[0], w[1]};
  };
  if (len <= 0) {  // no keys: a zero row, written once
    if (split == 0) store(O);
    return;
  }
  if (kbeg >= len) return;
  const int ns = min((len + kAttnSplit - 1) / kAttnSplit, max_splits);
  float M = -INFINITY;
  for (int w = 0; w < np; ++w) M = fmaxf(M, m_lds[w][m]);
  float L = 0.f;
  for (int w = 0; w < np; ++w) {
    const float mw = m_lds[w][m];
    const float f = (mw == -INFINITY) ? 0.f : exp2f(mw - M);
#pragma unroll
    for (int e = 0; e < NB; e += 4) {
      const f32x4 ow = *reinterpret_cast<const f32x4*>(&o_lds[w][m][d + e]);
#pragma unroll
      for (int c = 0; c < 4; ++c) O[e + c] = fmaf(ow[c], f, O[e + c]);
    }
    L = fmaf(l_lds[w][m], f, L);
  }
#pragma unroll
  for (int e = 0; e < NB; ++e) O[e] += np < NP ? 0.f : -0.f;  // parts without keys add +0, others nothing
  if (ns == 1) {
    const float f = (M == -INFINITY) ? 0.f : exp2f(M - M);
#pragma unroll
    for (int e = 0; e < NB; ++e) O[e] = attn_finish(fmaf(O[e], f, 0.f), fmaf(L, f, 0.f));
    store(O);
  } else {
    const int64_t pidx = oh * max_splits + split;
#pragma unroll
    for (int e = 0; e < NB; e += 4)
      *reinterpret_cast<f32x4*>(part_o + pidx * DH + d + e) = f32x4{O[e], O[e + 1], O[e + 2], O[e + 3]};
    if (d == 0) {
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
