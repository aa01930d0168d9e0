// Full-sequence (prefill) side of the low-rank RoPE attention, split the way a 288 GB part wants it:
//
//  1. lowrank_expand_kernel — Y = P @ u^T on the matrix cores for all tokens at once, with the head
//     epilogue fused: bias, rotate-half RoPE at the token's absolute position, and a strided store
//     straight into its destination (the query buffer [B,M,H,dh], or the dense KV cache rows
//     [B,S,Hk,dh] the decode kernels read later).  Both MFMA operands are contiguous along the rank
//     axis (P rows, nn.Linear-layout u rows), so they are plain 16-byte global loads in the
//     instruction's native lane layout; a wave owns 32 tokens x 128 head columns (16 accumulator
//     tiles) and d / d+64 of a head sit in the same lane, which keeps the rotation register-local.
//     K and V are rebuilt exactly once per token (the reference's fused kernel rebuilds every key
//     tile once per query tile to avoid the HBM round trip; with 288 GB that trade goes the other way).
//
//  2. attn_prefill_kernel — causal flash attention over the rotated q and the cache rows, transposed (S^T = K Q^T,
//     O^T = V^T P^T) on MFMA 16x16x32, online softmax in fp32 on the accumulator layout, the weights as a 16-bit high part
//     plus a 16-bit residual.  Key padding mask, additive mask and "fully masked row -> 0" follow the reference kernel.
#include "common.hpp"
#include "kernels.hpp"

namespace fsvd {

constexpr int kPfThreads = 256;

// eight elements as a matrix-core operand (F = the element type's fragment)
template <class F>
__device__ __forceinline__ F pf_ld(const uint16_t* p) {
  return __builtin_bit_cast(F, *reinterpret_cast<const u32x4_t*>(p));
}
template <class F>
__device__ __forceinline__ F pf_zero() { return __builtin_bit_cast(F, u32x4_t{0u, 0u, 0u, 0u}); }

// ---------------------------------------------------------------------------------------------
// 1. Y[token, head, :] = epilogue( P[token, (head), :] @ u[head*128 + :, :]^T )
//    grid (ceil(T/128), heads), 4 waves x 32 tokens
// ---------------------------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(kPfThreads) void lowrank_expand_kernel(ExpandArgs a) {
  typedef E16<DT> E;
  typedef typename E::frag_t frag_t;
  constexpr int DH = 128, NT = 8, HALF = 64;
  const int head = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  const int T = a.B * a.M;
  const int row0 = blockIdx.x * 128 + wave * 32;
  if (row0 >= T) return;

  const uint16_t* arow[2];
#pragma unroll
  for (int mi = 0; mi < 2; ++mi) {
    const int r = min(row0 + mi * 16 + lr, T - 1);
    const int b = r / a.M, m = r % a.M;
    arow[mi] = a.p + (int64_t)b * a.sp_b + (int64_t)m * a.sp_m + (int64_t)head * a.sp_h + lg * 8;
  }
  const uint16_t* brow = a.u + (int64_t)(head * DH + lr) * a.ldu + lg * 8;

  f32x4_t acc[2][NT];
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[mi][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
  for (int r0 = 0; r0 < a.R; r0 += 32) {
    const bool in = r0 + lg * 8 < a.R;
    frag_t af[2], bf[NT];
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) af[mi] = in ? pf_ld<frag_t>(arow[mi] + r0) : pf_zero<frag_t>();
#pragma unroll
    for (int t = 0; t < NT; ++t) bf[t] = in ? pf_ld<frag_t>(brow + (int64_t)t * 16 * a.ldu + r0) : pf_zero<frag_t>();
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[mi][t] = E::mfma(af[mi], bf[t], acc[mi][t]);
  }

  // epilogue on the accumulator layout: lane holds rows lg*4+i, column t*16+lr of each tile
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = row0 + mi * 16 + lg * 4 + i;
      if (r >= T) continue;
      const int b = r / a.M, m = r % a.M;
      const int pos = (a.positions ? a.positions[b] : a.pos0) + m;
      float x[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        float v = acc[mi][t][i];
        if (a.bias) v += E::val(a.bias[head * DH + t * 16 + lr]);
        x[t] = E::rnd(v);                       // the projection's own rounding point
      }
      if (a.cos) {
        // eager bf16 arithmetic: x0*c - x1*s and x1*c + x0*s, one rounding per op
        const int tp = min(max(pos, 0), a.rope_len - 1);
#pragma unroll
        for (int t = 0; t < NT / 2; ++t) {
          const float c = E::val(a.cos[(int64_t)tp * HALF + t * 16 + lr]);
          const float s = E::val(a.sin[(int64_t)tp * HALF + t * 16 + lr]);
          const float x0 = x[t], x1 = x[t + NT / 2];
          x[t] = E::rnd(E::rnd(x0 * c) - E::rnd(x1 * s));
          x[t + NT / 2] = E::rnd(E::rnd(x1 * c) + E::rnd(x0 * s));
        }
      }
      const int slot = a.dst_by_position ? pos : m;
      if (slot < 0 || slot >= a.dst_rows) continue;   // outside the destination: dropped
      uint16_t* dst = a.y + (int64_t)b * a.sy_b + (int64_t)slot * a.sy_m + (int64_t)head * a.sy_h;
#pragma unroll
      for (int t = 0; t < NT; ++t) dst[t * 16 + lr] = (uint16_t)E::bits(x[t]);
    }
}

// ---------------------------------------------------------------------------------------------
// 2. causal flash attention, head_dim 128: 32, 64 or 128 queries per workgroup (16 MI per wave), K and V tiles shared
//     through LDS.  With every wave fetching its own K fragments a 64-key tile costs 80 KB of L2 traffic per 64
//     queries and the kernel is bound by L2 requests; here a tile is read ONCE per workgroup, coalesced, one tile
//     ahead into registers, and written to LDS (K row-major with a padded stride, V transposed: four adjacent keys
//     per 8-byte write, rows of 128 bytes whose 16-byte pieces are XOR-ed with (d / 2 % 8) ^ (d / 8 % 8): the 16-byte
//     fragment reads — served 16 lanes a cycle, lanes 0-3, 12-15, 20-27 / 4-11, 16-19, 28-31 of a half wave — and the
//     8-byte transposing writes, 8 lanes a cycle, then both touch every bank once; found by enumeration).
//
//     Scores are computed TRANSPOSED, S^T = K Q^T: an accumulator lane then holds four consecutive keys of ONE query
//     (column lr), so the softmax statistics are one value per lane and query block, and the eight softmax weights a
//     lane owns in two 16-key blocks are exactly one B-operand fragment of O^T = V^T P^T — P never goes through LDS.
//     The price is a key order inside every 32 keys that the V tile has to follow: MFMA k-slot (lg, e) holds key
//     16 (e / 4) + 4 lg + e % 4, so V^T is stored with key offset ko at column 8 (ko % 16 / 4) + 4 (ko / 16) + ko % 4.
//     P is a bf16 high part plus a bf16 residual (two products per fragment) so that it carries ~16 mantissa bits.
//
//     A 64-key tile is 1536 cycles of products per 32 queries, and the vector work between them is as long, so every
//     instruction per score counts: tiles without masked keys test nothing, maxima and sums cross the four lanes of a query
//     by register swaps, the output is rescaled only in tiles that raise a maximum (a multiplication by one otherwise),
//     roundings are packed two to an instruction, and the key padding mask is one 64-bit word per tile: a tile without a
//     masked key runs unmasked, one without a visible key is skipped.  All of it gives the bits of the plain
//     formula (one multiply-add in front of the exponential instruction and row sums left to the end would save another 4 %).
//     Measured before -> after: 8 x 2048 tokens of 32 heads 758 -> 602 us, 4 x 1024 tokens 161 -> 122, with a
//     padding mask 215 -> 120; 512 tokens 19.0 -> 16.0.  Then, with every XCD starting the long tiles of all its heads first instead of
//     head by head (on average 1.2 of two possible waves were resident per SIMD): 576 -> 506 us (543 TFLOP/s), 122 -> 85, padded
//     121 -> 83; one sequence of 1024 / 2048 tokens 43 -> 36, 121 -> 97, 700 behind 1000 72 -> 63.  Below 128 rows a kernel without shared
//     tiles ran: two chunks of 77 rows behind 1411 tokens (32 / 8 heads) 181 -> 31 us, with 32 rows per workgroup 25.6.  Two LDS stages instead of one, raised
//     priority around the products and scalar address parts were built and gave nothing: two workgroups share a compute
//     unit, and each covers the other's waits.
// ---------------------------------------------------------------------------------------------
// the other lanes' values of a column (lane % 16) by register swaps: the largest of the four, and their sum
__device__ __forceinline__ float column_max(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const float w = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  const uint32_t x = __float_as_uint(w);
  const auto q = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}
__device__ __forceinline__ float column_sum(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const uint32_t x = __float_as_uint(__uint_as_float(r[0]) + __uint_as_float(r[1]));
  const auto q = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}
// exp(s * scale - m), every step rounded by itself
__device__ __forceinline__ float weight_of(float s, float scale, float m) {
#pragma clang fp contract(off)
  const float v = s * scale;
  return __expf(v - m);
}

// NG > 1: NG groups of four waves, each with K / V tiles of its own, take every NG-th key tile, and their running
// statistics and outputs are merged through LDS at the end — for calls whose (query tile, head) pairs number no more than
// the compute units, where a workgroup alone on its compute unit walks its key tiles with one wave per SIMD and waits out
// every load and barrier.
// NW: waves of a group, 16 MI query rows each (see launch_prefill_attn_t).
template <int DT, int MI, int NG, int NW>
__global__ __launch_bounds__(kWave * NW * NG, NG == 1 ? 2 : 1) void attn_prefill_kernel(PrefillAttnArgs a) {
  typedef E16<DT> E;
  typedef typename E::frag_t frag_t;
  constexpr int DH = 128, BN = 64, QW = 16 * MI, BM = NW * QW, VSTR = BN;
  constexpr int TG = kWave * NW, SR = TG / 16, PASS = BN / 4 / SR;   // threads of a group; rows that it stages at a time; passes over V's 16 groups of four keys
  // K rows of 288 bytes: a 16-byte LDS read is served 16 lanes a cycle (lanes 0-3, 12-15, 20-27 / 4-11, 16-19, 28-31 of a
  // half wave); rows 16 r apart with r odd multiples of 32 bytes give those lanes 16 different bank groups
  constexpr int KSTR = DH + 16;
  extern __shared__ __align__(16) unsigned char pw_smem[];
  constexpr int kGroupBytes = BN * KSTR * 2 + DH * VSTR * 2;
  const int grp = NG == 1 ? 0 : (int)threadIdx.x / TG;
  unsigned char* gsm = pw_smem + (size_t)grp * kGroupBytes;
  uint16_t (*Ks)[KSTR] = reinterpret_cast<uint16_t (*)[KSTR]>(gsm);                                   // [BN][KSTR]
  uint16_t (*Vt)[VSTR] = reinterpret_cast<uint16_t (*)[VSTR]>(gsm + (size_t)BN * KSTR * 2);            // [DH][VSTR]

  // The query tiles of a head (and the heads of a kv head) run on one XCD, so its K and V come out of one L2; the sequences of
  // a batch, which padding makes unequal, are spread over all of them.  Under a causal mask the last tiles see the most keys:
  // every XCD starts those of all its heads first, so that the short ones fill the end of the launch, and the tiles of a head
  // walk its keys side by side.
  const int MT = gridDim.x, HB = gridDim.y * gridDim.z, id = blockIdx.x + MT * (blockIdx.y + gridDim.y * blockIdx.z);
  int mt, hb;
  if (HB % 8 == 0) {
    const int per = HB >> 3, r = id >> 3;
    mt = r / per;
    hb = (id & 7) * per + r - mt * per;
  } else {
    const int t = xcd_run_index(id, MT * HB);
    hb = t / MT;
    mt = t - hb * MT;
  }
  if (a.causal) mt = MT - 1 - mt;
  const int h = hb / (int)gridDim.z, b = hb - h * (int)gridDim.z;
  const int hk = h / (a.H / a.Hk);
  const int tid = threadIdx.x % TG, lane = tid & 63, wave = tid >> 6;   // thread and wave within the group
  const int lr = lane & 15, lg = lane >> 4;
  const int q0 = a.q_pos0 ? a.q_pos0[b] : a.pos0;
  const int m_base = mt * BM + wave * QW;
  const int n_keys_all = max(1, min(q0 + a.M, a.S));

  frag_t qf[MI][4];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const int m = min(m_base + mi * 16 + lr, a.M - 1);
    const uint16_t* qp = a.q + (int64_t)b * a.sq_b + (int64_t)m * a.sq_m + (int64_t)h * a.sq_h + lg * 8;
#pragma unroll
    for (int st = 0; st < 4; ++st) qf[mi][st] = pf_ld<frag_t>(qp + st * 32);
  }
  float m_run[MI], l_run[MI];          // statistics of query m_base + 16 mi + lr (the same in the four lanes lg of a column)
  f32x4_t o[MI][8];                    // O^T: tile t, element i = dimension 16 t + 4 lg + i of that query
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    m_run[mi] = -INFINITY; l_run[mi] = 0.f;
#pragma unroll
    for (int t = 0; t < 8; ++t) o[mi][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  const int last_m = min(mt * BM + BM - 1, a.M - 1);
  const int k_end = a.causal ? min(n_keys_all, q0 + last_m + 1) : n_keys_all;
  // last key this wave's rows may see: tiles past it are skipped by the wave (it still takes part in the staging)
  const int wave_end = m_base >= a.M ? 0 : (a.causal ? min(n_keys_all, q0 + min(m_base + QW - 1, a.M - 1) + 1) : n_keys_all);
  const uint16_t* kb = a.k + (int64_t)b * a.sk_b + (int64_t)hk * a.sk_h;
  const uint16_t* vb = a.v + (int64_t)b * a.sk_b + (int64_t)hk * a.sk_h;
  // the maximum is taken of the unscaled scores; an additive mask and a scale that does not keep the order take the long way
  const bool direct = a.add_mask == nullptr && a.scale > 0.f;

  // staging roles: 16 lanes cover one 256-byte row; K: rows tid/16 + SR j; V: the four adjacent keys 4 (tid/16 + SR p) + j
  const int srow = tid >> 4, d0 = (tid & 15) * 8;
  // column of this thread's four keys in the permuted order of V^T (see above), before the bank swizzle
  const auto vcol_of = [](int row4) {
    const int vko = (row4 * 4) & 31;
    return ((row4 * 4) & 32) + 8 * ((vko & 15) >> 2) + 4 * (vko >> 4);
  };
  u32x4_t kreg[4 * PASS], vreg[4 * PASS];
  // the padding mask of a key tile travels with it: its bytes requested with the tile (the group's first wave, one key per
  // lane), parked in LDS beside it as one word, bit = key
  __shared__ uint64_t pms[NG];
  uint8_t pmreg = 1;
  auto request = [&](int n0) {
#pragma unroll
    for (int j = 0; j < 4 * PASS; ++j) {
      const int kkey = min(n0 + srow + SR * j, n_keys_all - 1), vkey = min(n0 + (srow + SR * (j >> 2)) * 4 + (j & 3), n_keys_all - 1);
      kreg[j] = *reinterpret_cast<const u32x4_t*>(kb + (int64_t)kkey * a.sk_s + d0);
      vreg[j] = *reinterpret_cast<const u32x4_t*>(vb + (int64_t)vkey * a.sk_s + d0);
    }
    if (a.pad_mask && tid < BN) pmreg = a.pad_mask[(int64_t)b * a.spm_b + min(n0 + tid, n_keys_all - 1)];
  };
  if (grp * BN < k_end) request(grp * BN);

  for (int n00 = 0; n00 < k_end; n00 += NG * BN) {
    const int n0 = n00 + grp * BN;
    const bool live = n0 < k_end;       // a group may have no tile in the last round; it still meets the barriers
    __syncthreads();   // the previous tile's Ks / Vt are consumed
    if (live) {
    if (a.pad_mask && tid < BN) {
      const uint64_t seen = __ballot(pmreg != 0);
      if (tid == 0) pms[grp] = seen;
    }
#pragma unroll
    for (int j = 0; j < 4 * PASS; ++j) *reinterpret_cast<u32x4_t*>(&Ks[srow + SR * j][d0]) = kreg[j];
#pragma unroll
    for (int p = 0; p < PASS; ++p) {
      const u32x4_t *v = vreg + 4 * p;
      const int vcol = vcol_of(srow + SR * p);
      const uint32_t w[4][4] = {{v[0].x, v[0].y, v[0].z, v[0].w}, {v[1].x, v[1].y, v[1].z, v[1].w},
                                {v[2].x, v[2].y, v[2].z, v[2].w}, {v[3].x, v[3].y, v[3].z, v[3].w}};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        u32x2_t lo, hi;   // dimensions d0 + 2c (low halves) and d0 + 2c + 1 (high halves) of the four keys
        lo.x = __builtin_amdgcn_perm(w[1][c], w[0][c], 0x05040100u);
        lo.y = __builtin_amdgcn_perm(w[3][c], w[2][c], 0x05040100u);
        hi.x = __builtin_amdgcn_perm(w[1][c], w[0][c], 0x07060302u);
        hi.y = __builtin_amdgcn_perm(w[3][c], w[2][c], 0x07060302u);
        // rows d0 + 2c and d0 + 2c + 1 share the swizzle term (row / 2 % 8) ^ (row / 8 % 8)
        const int col = vcol ^ (8 * (((((tid & 1) << 2) + c) ^ (tid & 7))));
        *reinterpret_cast<u32x2_t*>(&Vt[d0 + 2 * c][col]) = lo;
        *reinterpret_cast<u32x2_t*>(&Vt[d0 + 2 * c + 1][col]) = hi;
      }
    }
    }
    __syncthreads();   // tile visible
    if (n0 + NG * BN < k_end) request(n0 + NG * BN);
    if (!live || n0 >= wave_end) continue;   // nothing this wave's rows may see (wave-uniform)
    uint64_t seen = ~0ull;                   // keys of the tile that the padding mask leaves
    if (a.pad_mask) {
      const uint64_t w = pms[grp];
      seen = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)w) | ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(w >> 32)) << 32);
      if (seen == 0) continue;
    }

    // ---- S^T = K Q^T for 64 keys x 16 MI queries: block j, element i = key n0 + 16 j + 4 lg + i, query column lr
    f32x4_t sacc[MI][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      frag_t kf[4];
#pragma unroll
      for (int st = 0; st < 4; ++st) kf[st] = pf_ld<frag_t>(&Ks[j * 16 + lr][st * 32 + lg * 8]);
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        sacc[mi][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < 4; ++st) sacc[mi][j] = E::mfma(kf[st], qf[mi][st], sacc[mi][j]);
      }
    }
    // ---- masks + online softmax, one query per lane and block; tiles that need no mask take the short way
    const bool plain = seen == ~0ull && n0 + BN <= n_keys_all && (!a.causal || n0 + BN - 1 <= q0 + m_base);
    frag_t ph[MI][2], pl[MI][2];     // P^T fragments (high part, residual) of the two 32-key steps
    const uint64_t mine = seen >> (4 * lg);  // bit 16 j + i: key n0 + 16 j + 4 lg + i
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      const int m = m_base + mi * 16 + lr;
      const int vis = min(n_keys_all, a.causal ? q0 + m + 1 : n_keys_all) - n0 - lg * 4;   // keys of this lane's first block that exist for it, and so on
      if (!plain && seen == ~0ull) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) sacc[mi][j][i] = j * 16 + i < vis ? sacc[mi][j][i] : -INFINITY;
      } else if (!plain) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const bool ok = j * 16 + i < vis && ((mine >> (16 * j + i)) & 1) != 0;
            if (!ok) sacc[mi][j][i] = -INFINITY;       // mask first, then the additive term, as the reference kernel
          }
      }
      if (!direct) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const bool ok = plain || (j * 16 + i < vis && ((mine >> (16 * j + i)) & 1) != 0);
            float v = -INFINITY;
            if (ok) {
              v = sacc[mi][j][i] * a.scale;
              if (a.add_mask && m < a.M) v += a.add_mask[(int64_t)b * a.sam_b + (int64_t)m * a.sam_q + n0 + j * 16 + lg * 4 + i];
            }
            sacc[mi][j][i] = v;
          }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sacc[mi][j][i]);
      mx = column_max(mx);
      const float m_old = m_run[mi];
      const float m_new = fmaxf(m_old, direct ? mx * a.scale : mx);
      float rsum = 0.f;
      if (direct) {
        const float m0 = m_new == -INFINITY ? 0.f : m_new;    // -inf (nothing seen yet) must not meet itself: exp(-inf - 0) = 0
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            sacc[mi][j][i] = weight_of(sacc[mi][j][i], a.scale, m0);
            rsum += sacc[mi][j][i];
          }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float v = sacc[mi][j][i];
            sacc[mi][j][i] = (v == -INFINITY || m_new == -INFINITY) ? 0.f : __expf(v - m_new);
            rsum += sacc[mi][j][i];
          }
      }
      rsum = column_sum(rsum);
      if (__any(m_new != m_old)) {           // wave-uniform
        const float alpha = m_old == -INFINITY ? 0.f : __expf(m_old - m_new);
        l_run[mi] = fmaf(l_run[mi], alpha, rsum);
#pragma unroll
        for (int t = 0; t < 8; ++t) o[mi][t] *= alpha;
        m_run[mi] = m_new;
      } else {
        l_run[mi] += rsum;
      }
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        uint32_t hw[4], lw[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {                  // k-slots 2c, 2c + 1: block 2 st + c / 2, elements 2 (c % 2), + 1
          const float x0 = sacc[mi][2 * st + (c >> 1)][2 * (c & 1)], x1 = sacc[mi][2 * st + (c >> 1)][2 * (c & 1) + 1];
          hw[c] = E::pack2(x0, x1);
          lw[c] = E::pack2(x0 - E::lo(hw[c]), x1 - E::hi(hw[c]));
        }
        ph[mi][st] = __builtin_bit_cast(frag_t, u32x4_t{hw[0], hw[1], hw[2], hw[3]});
        pl[mi][st] = __builtin_bit_cast(frag_t, u32x4_t{lw[0], lw[1], lw[2], lw[3]});
      }
    }
    // ---- O^T += V^T P^T : A = Vt rows (dimension 16 t + lr; keys in the permuted order), B = P^T fragments
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const frag_t vf = pf_ld<frag_t>(&Vt[t * 16 + lr][(st * 32 + lg * 8) ^ (8 * ((lr >> 1) ^ ((2 * t + (lr >> 3)) & 7)))]);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
          o[mi][t] = E::mfma(vf, ph[mi][st], o[mi][t]);
          o[mi][t] = E::mfma(vf, pl[mi][st], o[mi][t]);
        }
      }
    }
  }
  if (NG > 1) {
    // merge the groups: (m, l, O) of groups 1.. through LDS (word-major, one 16-byte word per lane and slot)
    f32x4_t* mb = reinterpret_cast<f32x4_t*>(pw_smem);
    __syncthreads();                   // all groups are done with their K / V tiles
    if (grp > 0) {
      f32x4_t* mg = mb + (size_t)(grp - 1) * MI * 9 * TG;
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        mg[(mi * 9) * TG + tid] = f32x4_t{m_run[mi], l_run[mi], 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 8; ++t) mg[(mi * 9 + 1 + t) * TG + tid] = o[mi][t];
      }
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int g = 0; g < NG - 1; ++g) {
      const f32x4_t* mg = mb + (size_t)g * MI * 9 * TG;
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        const f32x4_t st = mg[(mi * 9) * TG + tid];
        const float m1 = st[0], l1 = st[1];
        const float m = fmaxf(m_run[mi], m1);
        const float a0 = m_run[mi] == -INFINITY ? 0.f : __expf(m_run[mi] - m), a1 = m1 == -INFINITY ? 0.f : __expf(m1 - m);
        l_run[mi] = l_run[mi] * a0 + l1 * a1;
        m_run[mi] = m;
#pragma unroll
        for (int t = 0; t < 8; ++t) o[mi][t] = o[mi][t] * a0 + mg[(mi * 9 + 1 + t) * TG + tid] * a1;
      }
    }
  }
  // ---- normalise and store (four consecutive dimensions per lane and tile, one 8-byte write where the destination
  // allows); rows with no visible key give 0
  const bool out8 = (reinterpret_cast<uintptr_t>(a.out) & 7) == 0 && (a.so_b % 4) == 0 && (a.so_m % 4) == 0 && (a.so_h % 4) == 0;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const int m = m_base + mi * 16 + lr;
    if (m >= a.M) continue;
    const float inv = l_run[mi] > 0.f ? 1.0f / l_run[mi] : 0.f;
    uint16_t* op = a.out + (int64_t)b * a.so_b + (int64_t)m * a.so_m + (int64_t)h * a.so_h + lg * 4;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const u32x2_t w{E::pack2(o[mi][t][0] * inv, o[mi][t][1] * inv), E::pack2(o[mi][t][2] * inv, o[mi][t][3] * inv)};
      if (out8) {
        *reinterpret_cast<u32x2_t*>(op + t * 16) = w;
      } else {
        op[t * 16] = (uint16_t)w.x; op[t * 16 + 1] = (uint16_t)(w.x >> 16);
        op[t * 16 + 2] = (uint16_t)w.y; op[t * 16 + 3] = (uint16_t)(w.y >> 16);
      }
    }
  }
}

// Rotation tables of given positions in one launch: cos and sin of position * inv_freq, rounded once.  As tensor operations (position
// to fp32, product, cosine, sine, two roundings) they were six launches of 2 to 6 us in front of an attention call of 240.
// A padding mask of whole numbers becomes the bytes that the attention reads in the same launch: the workgroups behind those of the
// tables compare it with zero, which as a tensor operation was a launch of 4.8 us (the call of 4 x 1024 tokens 200.6 -> 197.6 us).
template <int DT>
__global__ __launch_bounds__(256) void rope_tables_kernel(const int64_t* __restrict__ pos, const float* __restrict__ inv_freq, uint16_t* __restrict__ cos_out,
                                                          uint16_t* __restrict__ sin_out, int64_t n, int half, unsigned tables, const int64_t* __restrict__ mask,
                                                          uint8_t* __restrict__ pad, int64_t nmask) {
  typedef E16<DT> E;
  if (blockIdx.x >= tables) {
    const int64_t i = (int64_t)(blockIdx.x - tables) * 256 + threadIdx.x;
    if (i < nmask) pad[i] = mask[i] != 0;
    return;
  }
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float ang = (float)pos[i / half] * inv_freq[i % half];
  cos_out[i] = (uint16_t)E::bits(cosf(ang));
  sin_out[i] = (uint16_t)E::bits(sinf(ang));
}
int launch_rope_tables(const int64_t* pos, const float* inv_freq, uint16_t* cos_out, uint16_t* sin_out, int64_t rows, int half, const int64_t* mask,
                       uint8_t* pad, int64_t nmask, int dt, hipStream_t st) {
  const char* fn = "fsvd_rope_tables";
  constexpr int64_t kMost = (int64_t)0x3fffffff * 256;
  if (rows <= 0 || half <= 0 || rows > kMost * 2 / half || nmask < 0 || nmask > kMost) { set_last_error("%s: bad shape", fn); return kErrBadShape; }
  if (dt != 0 && dt != 1) { set_last_error("%s: dtype code %d (bf16 = 0 and fp16 = 1 are served)", fn, dt); return kErrBadDtype; }
  const unsigned tables = (unsigned)((rows * half + 255) / 256);
  const dim3 grid(tables + (unsigned)((nmask + 255) / 256));
  if (dt == 1) hipLaunchKernelGGL(rope_tables_kernel<1>, grid, dim3(256), 0, st, pos, inv_freq, cos_out, sin_out, rows * half, half, tables, mask, pad, nmask);
  else hipLaunchKernelGGL(rope_tables_kernel<0>, grid, dim3(256), 0, st, pos, inv_freq, cos_out, sin_out, rows * half, half, tables, mask, pad, nmask);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_last_error("%s: launch failed: %s", fn, hipGetErrorString(e)); return kErrLaunch; }
  return kOk;
}

int launch_expand(const ExpandArgs& a, hipStream_t st) {
  const char* fn = "fsvd_lowrank_expand_heads";
  if (a.dt != 0 && a.dt != 1) { set_last_error("%s: dtype code %d (bf16 = 0 and fp16 = 1 are served)", fn, a.dt); return kErrBadDtype; }
  if (a.B <= 0 || a.M <= 0 || a.heads <= 0 || a.R <= 0) { set_last_error("%s: empty shape", fn); return kErrBadShape; }
  if (a.Dh != 128) { set_last_error("%s: head_dim %d is not 128", fn, a.Dh); return kErrBadShape; }
  if (expand_tiles_apply(a)) return launch_expand_tiles(a, st);   // the LDS-tiled kernels
  if (a.R % 8) { set_last_error("%s: rank %d is not a multiple of 8 (coefficients of their own per head); pad the factors", fn, a.R); return kErrBadShape; }
  const auto mis = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) != 0; };
  if (mis(a.p) || mis(a.u) || (a.sp_b % 8) || (a.sp_m % 8) || (a.sp_h % 8) || (a.ldu % 8)) {
    set_last_error("%s: coefficient / factor pointers and strides must be 16-byte aligned", fn);
    return kErrBadAlign;
  }
  const int T = a.B * a.M;
  set_last_form("rows 128 heads");
  if (a.dt == 1) hipLaunchKernelGGL(lowrank_expand_kernel<1>, dim3((T + 127) / 128, a.heads), dim3(kPfThreads), 0, st, a);
  else hipLaunchKernelGGL(lowrank_expand_kernel<0>, dim3((T + 127) / 128, a.heads), dim3(kPfThreads), 0, st, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_last_error("%s: launch failed: %s", fn, hipGetErrorString(e)); return kErrLaunch; }
  return kOk;
}

template <int DT, int MI, int NG, int NW = 4>
static int launch_prefill_attn_form(const PrefillAttnArgs& a, hipStream_t st) {
  const char* fn = "fsvd_attn_prefill";
  constexpr size_t lds = (size_t)NG * ((size_t)64 * 144 * 2 + (size_t)128 * 64 * 2);
  if (NG > 1) {
    static bool granted = false;
    if (!granted) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_prefill_kernel<DT, MI, NG, NW>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) { set_last_error("%s: cannot reserve %zu bytes of LDS: %s", fn, lds, hipGetErrorString(e)); return kErrLaunch; }
      granted = true;
    }
  }
  hipLaunchKernelGGL((attn_prefill_kernel<DT, MI, NG, NW>), dim3((a.M + 16 * NW * MI - 1) / (16 * NW * MI), a.H, a.B), dim3(NG * NW * kWave), lds, st, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_last_error("%s: launch failed: %s", fn, hipGetErrorString(e)); return kErrLaunch; }
  return kOk;
}

template <int DT>
static int launch_prefill_attn_t(const PrefillAttnArgs& a, hipStream_t st) {
  // 128 query rows per workgroup from 1.5 workgroups per compute unit on, else 64 (half the rows per wave)
  const int64_t cu = compute_units();
  if ((int64_t)((a.M + 127) / 128) * a.H * a.B * 2 >= cu * 3) return launch_prefill_attn_form<DT, 2, 1>(a, st);
  // Fewer 64-row workgroups than compute units leave part of the chip idle, and one that has a compute unit to itself waits out every load and
  // barrier.  Where 32-row workgroups (two waves per group, the rest of the LDS for a fourth group) are one per compute unit at most, they:
  // us per call, 64 rows in three groups (two from 128 rows on) -> this: two chunks of 77 rows of 32 / 8 heads behind 1411 tokens 32.0 -> 25.6, one of
  // 40 behind 900 22.4 -> 18.9, 127 behind 1000 24.4 -> 19.0, 200 behind 1000 30.1 -> 22.6, two of 100 behind 500 17.3 -> 14.4, eight of 32 behind 400
  // (256 workgroups) 17.3 -> 15.9; one more round of them loses: two of 130 behind 300 (320 workgroups) 14.4 -> 18.8.  Three groups of them 29.3,
  // 20.4, 21.1, 25.3 at the first four; 16 rows and one wave per group no better at 40 rows, 46 at the first.  Four groups add the keys up in another
  // order than three: over 52 such calls of 17 to 7000 rows the error against 64 bits (0.0016 to 0.0017, the output's own rounding) changes by less than 5e-7 of itself.
  if ((int64_t)((a.M + 31) / 32) * a.H * a.B <= cu) return launch_prefill_attn_form<DT, 1, 4, 2>(a, st);
  // Up to ~1.5 of 64 rows: three groups of waves share a workgroup's key tiles below 128 rows (four spill), two from there on: 512 rows of 32 heads
  // (256 workgroups) 18.0 / 15.9 / 15.4 us with one / two / three groups, 700 rows (352) 23.7 / 20.3 / 19.1, 1024 rows (512) 37.3 / 38.9 / 37.7.  The
  // half microsecond that the third would give there (0.2 % of a prompt pass of 32 layers) does not pay for another order of the sums: the
  // layers hand a flipped rounding on until the logits of 512 rows end 0.04 (relative) from the present ones.
  const int64_t tiles = (int64_t)((a.M + 63) / 64) * a.H * a.B;
  if (tiles <= cu && a.M < 128) return launch_prefill_attn_form<DT, 1, 3>(a, st);
  if (tiles * 2 <= cu * 3) return launch_prefill_attn_form<DT, 1, 2>(a, st);
  return launch_prefill_attn_form<DT, 1, 1>(a, st);
}

int launch_prefill_attn(const PrefillAttnArgs& a, hipStream_t st) {
  const char* fn = "fsvd_attn_prefill";
  if (a.dt != 0 && a.dt != 1) { set_last_error("%s: dtype code %d (bf16 = 0 and fp16 = 1 are served)", fn, a.dt); return kErrBadDtype; }
  if (a.B <= 0 || a.M <= 0 || a.H <= 0 || a.Hk <= 0 || a.H % a.Hk) { set_last_error("%s: bad shape", fn); return kErrBadShape; }
  if (a.Dh != 128) { set_last_error("%s: head_dim %d is not 128", fn, a.Dh); return kErrBadShape; }
  const auto mis = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) != 0; };
  if (mis(a.q) || mis(a.k) || mis(a.v) || (a.sq_b % 8) || (a.sq_m % 8) || (a.sq_h % 8) || (a.sk_b % 8) || (a.sk_s % 8) || (a.sk_h % 8)) {
    set_last_error("%s: q / k / v pointers and strides must be 16-byte aligned", fn);
    return kErrBadAlign;
  }
  return a.dt == 1 ? launch_prefill_attn_t<1>(a, st) : launch_prefill_attn_t<0>(a, st);
}

}  // namespace fsvd
