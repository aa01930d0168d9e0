// Single-query attention over a dense KV cache [B,S,Hk,Dh] (K stored post-RoPE), split over
// the key axis so that B*H*nsplit workgroups cover the chip.  Each workgroup scores its key
// range in passes of 128 keys: every K and V row of a pass is requested up front (16-byte loads,
// 16 in flight per lane), scores come from V_DOT2 against the query chunk held in registers with
// a DPP fold over the lanes that share a key, the softmax is the online (running max / sum)
// form and p*V accumulates per lane.  The workgroup writes an un-normalised partial (acc, m, l)
// with write-through stores; the last workgroup to arrive for a (b,h) merges the partials in
// split order, so the result does not depend on arrival order.
#include "common.hpp"
#include "kernels.hpp"

namespace fsvd {

constexpr int kAttnThreads = 256;
// cache rows for each range that the caller has scratch for: a bound on what a call may ask, not on what a workgroup walks (a
// sequence may be cut into fewer ranges than that, decode_map.hpp; the key loop is streamed)
constexpr int kMaxRowsPerRange = 1 << 20;

// The range, head (or head group, H of them) and sequence of this workgroup, len = seqlens[b] and the number of ranges of that
// sequence.  Five to 64 sequences: a wave has all their lengths, and all workgroups come to the same assignment.  Up to four take the
// first ranges first whatever their lengths (what the lengths would tell comes 0.2 us later, 3 percent of 129 keys), as long as that leaves
// the heads of a kv head together (28 heads over four, 1500 keys 11.7 -> 14.1).
__device__ __forceinline__ int decode_keys(const AttnDecodeArgs& a, int len) { return max(0, min(len + a.seqlen_add, a.S)); }
__device__ __forceinline__ void decode_work_item(const AttnDecodeArgs& a, int H, int& b, int& h, int& s, int& len, int& ranges) {
  DecodeSlot slot;
  asm volatile("" :: "s"(a.q), "s"(a.seqlen_add));   // the lines of the arguments that are needed behind the lengths, along with the others
  int one_below = a.plan.one_below;
  const bool sorts = a.plan.by_length > 0.f;
  if (a.B > 4 && a.B <= 64 && (a.nsplit > 1 || sorts)) {
    const int lane = threadIdx.x & 63, n = a.seqlens[min(lane, a.B - 1)];     // lanes past the last sequence repeat it
    slot = decode_slot_by_range(blockIdx.x, a.B, H, a.nsplit);
    asm volatile("" : "+s"(slot.s), "+s"(slot.h), "+s"(slot.seq));      // the divisions while the lengths are on their way
    const int keys = decode_keys(a, n);
    const auto any_from = [&](int k) { return __ballot(keys >= k) != 0; };
    const float uneven = any_from(kDecodeLong) ? a.plan.by_length : (any_from(kDecodeShort) ? a.plan.by_length_short : 0.f);
    if (any_from(one_below)) one_below = 0;
    bool by_length = uneven == kDecodeAlways;
    if ((sorts && uneven > kDecodeAlways) || (one_below > 0 && a.plan.one_if_even)) {
      const float longest = wave_max((float)keys), mean = wave_sum(lane < a.B ? (float)keys : 0.f) / a.B;
      if (a.plan.one_if_even && longest > 1.5f * mean) one_below = 0;
      by_length |= uneven > 0.f && longest > uneven * mean;
    }
    if (by_length) {
      slot = decode_slot_by_length(blockIdx.x, a.B, H, a.nsplit);
      int rank = 0;                     // of this lane's sequence, longest first
      for (int u = 0; u < a.B; ++u) {
        const int nu = __builtin_amdgcn_readlane(n, u);
        rank += nu > n || (nu == n && u < lane);
      }
      slot.seq = __builtin_ctzll(__ballot(lane < a.B && rank == slot.seq));
    } else if (one_below > 0 || !any_from(128 * (a.nsplit >> 1) + 1)) {          // at least half of the ranges have no keys
      slot = decode_slot_by_pair(blockIdx.x, a.B, H, a.nsplit);
    }
    len = __builtin_amdgcn_readlane(n, slot.seq);
  } else {
    slot = (a.B <= 4 && a.B * H % 8 == 0) || one_below > 0 ? decode_slot_by_pair(blockIdx.x, a.B, H, a.nsplit) : decode_slot_by_range(blockIdx.x, a.B, H, a.nsplit);
    len = a.seqlens[slot.seq];
  }
  b = slot.seq;
  h = slot.h;
  s = slot.s;
  ranges = decode_ranges(one_below, a.nsplit, decode_keys(a, len));
}

// coherent (L2-bypassing) scalar accessors for the cross-workgroup partials: the producers write
// through to memory and the merging workgroup reads from memory, so no L2 write-back / invalidate
// fence is needed (those serialise per XCD and cost more than the whole kernel)
__device__ __forceinline__ void st_agent(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float ld_agent(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// dimensions d and d + half of the new row of (b, hk): k_new rotated at position pos (fp32 math, one rounding), v_new as it is
template <int DT, class Args>
__device__ __forceinline__ void append_pair(const Args& a, int half, int b, int hk, int pos, int d) {
  typedef E16<DT> E;
  const uint16_t* kp = a.k_new + (int64_t)b * a.sk_b + (int64_t)hk * a.sk_h;
  const uint16_t* vp = a.v_new + (int64_t)b * a.sv_b + (int64_t)hk * a.sv_h;
  float x0 = E::val(kp[d]), x1 = E::val(kp[d + half]);
  if (a.cos) {
    const int tp = min(pos, a.rope_len - 1);
    const float c = E::val(a.cos[(int64_t)tp * half + d]);
    const float s = E::val(a.sin[(int64_t)tp * half + d]);
    const float r0 = x0 * c - x1 * s, r1 = x0 * s + x1 * c;
    x0 = r0; x1 = r1;
  }
  const int64_t off = (int64_t)b * a.sc_b + (int64_t)pos * a.sc_s + (int64_t)hk * a.sc_h;
  uint16_t* kc = const_cast<uint16_t*>(a.k_cache) + off;
  uint16_t* vc = const_cast<uint16_t*>(a.v_cache) + off;
  kc[d] = (uint16_t)E::bits(x0);
  kc[d + half] = (uint16_t)E::bits(x1);
  vc[d] = vp[d];
  vc[d + half] = vp[d + half];
}

// The new row of a sequence is its last key: the workgroup whose keys [k0, k1) end with it writes it before it reads them.
// Only where no other workgroup reads the row (launch_attn_decode).  Against a launch of its own for the append: 16 sequences of
// up to 4001 keys, 32 heads over 8, 53.5 -> 50.1 us, 64 x 1000 49.8 -> 48.0, 16 x 1000 with 32 kv heads 49.6 -> 46.9.
template <int DT, int DH>
__device__ __forceinline__ void append_own_row(const AttnDecodeArgs& a, int b, int hk, int pos, int k0, int k1) {
  if (a.k_new == nullptr) return;
  if (pos < k0 || pos >= k1) return;               // the same for the whole workgroup; k1 <= S
  if (threadIdx.x < DH / 2) append_pair<DT>(a, DH / 2, b, hk, pos, threadIdx.x);
  wait_stores_acked();
  __syncthreads();
}

// (head_dim 64 would fit eight waves on a SIMD, all of up to 2048 workgroups at once: 16 x 4000 keys of 32 heads 111.8 us, with seven 105.5)
// HALVES: caches that one pass covers and that are a single range (decode_one_pass): at most half a pass of keys takes half the loads.
template <int DT, int DH, int U, bool HALVES = false>
__global__ __launch_bounds__(kAttnThreads) __attribute__((amdgpu_waves_per_eu(1, DH == 64 ? 7 : 8))) void attn_decode_kernel(AttnDecodeArgs a) {
  typedef E16<DT> E;
  constexpr int LPK = DH / 8;                 // lanes that share one key (8 bf16 each)
  constexpr int KPB = kAttnThreads / LPK;     // keys per block pass
  constexpr int CH = KPB * U;                 // keys in flight per workgroup
  __shared__ __align__(16) float accs[KPB * DH];
  __shared__ __align__(16) uint16_t qs[DH];
  __shared__ float red[2][4];
  __shared__ int last_flag;

  int b, h, s, len, ranges;
  decode_work_item(a, a.H, b, h, s, len, ranges);
  if (s >= ranges) return;
  const int tid = threadIdx.x;
  const int hk = h / (a.H / a.Hk);
  const int n_keys = decode_keys(a, len);
  int per = (n_keys + ranges - 1) / ranges;
  per = (per + KPB - 1) / KPB * KPB;
  const int k0 = min(s * per, n_keys);
  const int k1 = min(n_keys, k0 + per);
  append_own_row<DT, DH>(a, b, hk, len, k0, k1);

  // query chunk (optionally rotated at position seqlens[b], fp32 math, one rounding)
  const uint16_t* qp = a.q + (int64_t)b * a.sq_b + (int64_t)h * a.sq_h;
  if (tid < DH / 2) {
    float x0 = E::val(qp[tid]), x1 = E::val(qp[tid + DH / 2]);
    if (a.cos) {
      const int tp = min(max(len, 0), a.rope_len - 1);
      const float c = E::val(a.cos[(int64_t)tp * (DH / 2) + tid]);
      const float sn = E::val(a.sin[(int64_t)tp * (DH / 2) + tid]);
      const float r0 = x0 * c - x1 * sn, r1 = x0 * sn + x1 * c;
      x0 = r0; x1 = r1;
    }
    qs[tid] = (uint16_t)E::bits(x0);
    qs[tid + DH / 2] = (uint16_t)E::bits(x1);
  }
  const int part = tid % LPK, slot = tid / LPK;
  const uint16_t* kbase = a.k_cache + (int64_t)b * a.sc_b + (int64_t)hk * a.sc_h + part * 8;
  const uint16_t* vbase = a.v_cache + (int64_t)b * a.sc_b + (int64_t)hk * a.sc_h + part * 8;

  float m_run = -INFINITY, l_thr = 0.f;
  float acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.f;
  const bool few = HALVES && k1 - k0 <= CH / 2;
  int it = 0;
  for (int c0 = k0; c0 < k1; c0 += CH, ++it) {
    // all K and V rows of this pass are requested before anything is consumed
    u32x4_t kv[U], vv[U];
    if constexpr (HALVES) {
#pragma unroll
      for (int u = U / 2; u < U; ++u) kv[u] = vv[u] = u32x4_t{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (few && u >= U / 2) break;
      const int key = min(c0 + u * KPB + slot, k1 - 1);
      kv[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(kbase + (int64_t)key * a.sc_s));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (few && u >= U / 2) break;
      const int key = min(c0 + u * KPB + slot, k1 - 1);
      vv[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(vbase + (int64_t)key * a.sc_s));
    }
    if (it == 0) __syncthreads();  // qs ready
    const u32x4_t qv = *reinterpret_cast<const u32x4_t*>(qs + part * 8);
    float sc[U];
    float lmax = -INFINITY;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float d = E::dot8(kv[u], qv, 0.f);
      d += dpp_f32<0xB1>(d);
      d += dpp_f32<0x4E>(d);
      d += dpp_f32<0x141>(d);
      if (LPK == 16) d += dpp_f32<0x140>(d);
      sc[u] = (c0 + u * KPB + slot < k1) ? d * a.scale : -INFINITY;
      lmax = fmaxf(lmax, sc[u]);
    }
    lmax = wave_max(lmax);
    const int rb = it & 1;
    if ((tid & 63) == 0) red[rb][tid >> 6] = lmax;
    __syncthreads();
    const float m_c = fmaxf(fmaxf(red[rb][0], red[rb][1]), fmaxf(red[rb][2], red[rb][3]));
    const float m_new = fmaxf(m_run, m_c);
    const float alpha = (m_run == -INFINITY) ? 0.f : __expf(m_run - m_new);
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] *= alpha;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float p = (sc[u] == -INFINITY) ? 0.f : __expf(sc[u] - m_new);
      psum += p;
      acc[0] += p * E::lo(vv[u].x); acc[1] += p * E::hi(vv[u].x);
      acc[2] += p * E::lo(vv[u].y); acc[3] += p * E::hi(vv[u].y);
      acc[4] += p * E::lo(vv[u].z); acc[5] += p * E::hi(vv[u].z);
      acc[6] += p * E::lo(vv[u].w); acc[7] += p * E::hi(vv[u].w);
    }
    l_thr = l_thr * alpha + (part == 0 ? psum : 0.f);
    m_run = m_new;
  }
  if (it == 0) __syncthreads();
  // fold the key slots and the per-thread sums
#pragma unroll
  for (int i = 0; i < 8; ++i) accs[slot * DH + part * 8 + i] = acc[i];
  float lw = wave_sum(l_thr);
  __syncthreads();  // red[] of the last pass consumed; accs written
  if ((tid & 63) == 0) red[0][tid >> 6] = lw;
  __syncthreads();
  const float l = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
  const float m = m_run;
  float o = 0.f;
  if (tid < DH) {
#pragma unroll 8
    for (int j = 0; j < KPB; ++j) o += accs[j * DH + tid];
  }

  uint16_t* outp = a.out + (int64_t)b * a.so_b + (int64_t)h * a.so_h;
  if (ranges == 1) {
    if (tid < DH) outp[tid] = (uint16_t)E::bits(l > 0.f ? o / l : 0.f);
    return;
  }
  float* part_ws = a.ws_part + ((int64_t)(b * a.H + h) * a.nsplit) * (DH + 2);
  float* mine = part_ws + (int64_t)s * (DH + 2);
  if (tid < DH) st_agent(mine + tid, o);
  if (tid == 0) { st_agent(mine + DH, m); st_agent(mine + DH + 1, l); }
  wait_stores_acked();
  __syncthreads();
  if (tid == 0) {
    const int old = __hip_atomic_fetch_add(&a.ws_count[b * a.H + h], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last_flag = (old == ranges - 1);
  }
  __syncthreads();
  if (!last_flag) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  if (tid < DH) {
    // the loads of eight splits are in flight at once (each comes from beyond this XCD's L2; one split per round trip
    // made this merge a third of the kernel at eight splits); the splits are added in order
    constexpr int SU = 8;
    float M = -INFINITY;
    for (int i0 = 0; i0 < ranges; i0 += SU) {
      float mi[SU];
#pragma unroll
      for (int u = 0; u < SU; ++u) mi[u] = ld_agent(part_ws + (int64_t)min(i0 + u, ranges - 1) * (DH + 2) + DH);
#pragma unroll
      for (int u = 0; u < SU; ++u) M = fmaxf(M, mi[u]);
    }
    float num = 0.f, den = 0.f;
    for (int i0 = 0; i0 < ranges; i0 += SU) {
      float mi[SU], oi[SU], li[SU];
#pragma unroll
      for (int u = 0; u < SU; ++u) {
        const float* pw = part_ws + (int64_t)min(i0 + u, ranges - 1) * (DH + 2);
        mi[u] = ld_agent(pw + DH);
        oi[u] = ld_agent(pw + tid);
        li[u] = ld_agent(pw + DH + 1);
      }
#pragma unroll
      for (int u = 0; u < SU; ++u) {
        const float w = (i0 + u >= ranges || mi[u] == -INFINITY) ? 0.f : __expf(mi[u] - M);
        num += w * oi[u];
        den += w * li[u];
      }
    }
    outp[tid] = (uint16_t)E::bits(den > 0.f ? num / den : 0.f);
  }
  if (tid == 0) __hip_atomic_store(&a.ws_count[b * a.H + h], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Grouped-query caches: G query heads of one kv head per workgroup.  The K and V rows of a pass are requested once and
// scored against the G queries (with one workgroup per query head every head of a group re-reads its kv head's rows from
// L2); running maximum, sum and accumulators per query head.  G divides H / Hk.
// At two workgroups per compute unit the vector work of G heads (about 900 instructions per wave and pass) is as long as
// the loads, so the two run at the same time: the K rows of a pass are replaced by the next pass's as soon as they are
// scored, the V rows as soon as they are added up.  The heads leave together: one fold through LDS, one arrival, one merge
// (head by head it was four hand-offs in a row).  Same bits.  With an append launch before it, 32 query heads over 8 kv heads:
// 16 x up to 4001 keys 61.4 -> 53.5 us (4.3 TB/s), 64 x 1000 52.9 -> 49.8, 40 x 1500 68.1 -> 65.1.
// Since then the loads' latency and the sequences' lengths bound it: with the scores on the matrix cores (40 % fewer instructions)
// 16 x up to 4001 keys took 50.3 us instead of 51.2, and 40 x 1500, read in pieces of 64 bytes, 77 instead of 64.
template <int DT, int DH, int U, int G>
__global__ __launch_bounds__(kAttnThreads) void attn_decode_gqa_kernel(AttnDecodeArgs a) {
  typedef E16<DT> E;
  constexpr int LPK = DH / 8, KPB = kAttnThreads / LPK, CH = KPB * U;
  static_assert(G * DH / 2 <= kAttnThreads, "one thread per rotation pair of every query of the group");
  __shared__ __align__(16) float accs[G][KPB * DH];
  __shared__ __align__(16) uint16_t qs[G][DH];
  __shared__ float red[2][4][G], sums[4][G];
  __shared__ int last_flag;

  int b, hg, s, len, ranges;
  decode_work_item(a, a.H / G, b, hg, s, len, ranges);
  if (s >= ranges) return;
  const int tid = threadIdx.x;
  const int h0 = hg * G, hk = h0 / (a.H / a.Hk);
  const int n_keys = decode_keys(a, len);
  int per = (n_keys + ranges - 1) / ranges;
  per = (per + KPB - 1) / KPB * KPB;
  const int k0 = min(s * per, n_keys);
  const int k1 = min(n_keys, k0 + per);
  append_own_row<DT, DH>(a, b, hk, len, k0, k1);

  if (tid < G * (DH / 2)) {
    const int g = tid / (DH / 2), d = tid % (DH / 2);
    const uint16_t* qp = a.q + (int64_t)b * a.sq_b + (int64_t)(h0 + g) * a.sq_h;
    float x0 = E::val(qp[d]), x1 = E::val(qp[d + DH / 2]);
    if (a.cos) {
      const int tp = min(max(len, 0), a.rope_len - 1);
      const float c = E::val(a.cos[(int64_t)tp * (DH / 2) + d]);
      const float sn = E::val(a.sin[(int64_t)tp * (DH / 2) + d]);
      const float r0 = x0 * c - x1 * sn, r1 = x0 * sn + x1 * c;
      x0 = r0; x1 = r1;
    }
    qs[g][d] = (uint16_t)E::bits(x0);
    qs[g][d + DH / 2] = (uint16_t)E::bits(x1);
  }
  const int part = tid % LPK, slot = tid / LPK;
  const uint16_t* kbase = a.k_cache + (int64_t)b * a.sc_b + (int64_t)hk * a.sc_h + part * 8;
  const uint16_t* vbase = a.v_cache + (int64_t)b * a.sc_b + (int64_t)hk * a.sc_h + part * 8;

  float m_run[G], l_thr[G], acc[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m_run[g] = -INFINITY; l_thr[g] = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[g][i] = 0.f;
  }
  u32x4_t kv[U], vv[U];
  const auto fetch = [&](u32x4_t (&r)[U], const uint16_t* base, int c0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int key = min(c0 + u * KPB + slot, k1 - 1);
      r[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(base + (int64_t)key * a.sc_s));
    }
  };
  if (k0 < k1) { fetch(kv, kbase, k0); fetch(vv, vbase, k0); }
  __syncthreads();  // qs ready
  int it = 0;
  for (int c0 = k0; c0 < k1; c0 += CH, ++it) {
    float sc[G][U];
    const int rb = it & 1;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const u32x4_t qv = *reinterpret_cast<const u32x4_t*>(&qs[g][part * 8]);
      float lmax = -INFINITY;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float d = E::dot8(kv[u], qv, 0.f);
        d += dpp_f32<0xB1>(d);
        d += dpp_f32<0x4E>(d);
        d += dpp_f32<0x141>(d);
        if (LPK == 16) d += dpp_f32<0x140>(d);
        sc[g][u] = (c0 + u * KPB + slot < k1) ? d * a.scale : -INFINITY;
        lmax = fmaxf(lmax, sc[g][u]);
      }
      lmax = wave_max(lmax);
      if ((tid & 63) == 0) red[rb][tid >> 6][g] = lmax;
    }
    // the K rows of the next pass are on their way during the softmax and P V of this one, its V rows during the scores
    // (past the last pass all lanes take the last key again: behind a condition the compiler would wait for the K rows
    // where it needs the V rows)
    __builtin_amdgcn_sched_barrier(0);
    fetch(kv, kbase, c0 + CH);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float m_c = fmaxf(fmaxf(red[rb][0][g], red[rb][1][g]), fmaxf(red[rb][2][g], red[rb][3][g]));
      const float m_new = fmaxf(m_run[g], m_c);
      const float alpha = (m_run[g] == -INFINITY) ? 0.f : __expf(m_run[g] - m_new);
      float psum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[g][i] *= alpha;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float p = (sc[g][u] == -INFINITY) ? 0.f : __expf(sc[g][u] - m_new);
        psum += p;
        acc[g][0] += p * E::lo(vv[u].x); acc[g][1] += p * E::hi(vv[u].x);
        acc[g][2] += p * E::lo(vv[u].y); acc[g][3] += p * E::hi(vv[u].y);
        acc[g][4] += p * E::lo(vv[u].z); acc[g][5] += p * E::hi(vv[u].z);
        acc[g][6] += p * E::lo(vv[u].w); acc[g][7] += p * E::hi(vv[u].w);
      }
      l_thr[g] = l_thr[g] * alpha + (part == 0 ? psum : 0.f);
      m_run[g] = m_new;
    }
    __builtin_amdgcn_sched_barrier(0);
    fetch(vv, vbase, c0 + CH);
    __builtin_amdgcn_sched_barrier(0);
  }
  // fold the key slots and the per-thread sums of all heads at once
#pragma unroll
  for (int g = 0; g < G; ++g) {
#pragma unroll
    for (int i = 0; i < 8; ++i) accs[g][slot * DH + part * 8 + i] = acc[g][i];
    const float lw = wave_sum(l_thr[g]);
    if ((tid & 63) == 0) sums[tid >> 6][g] = lw;
  }
  __syncthreads();
  // thread -> dimension tid % DH of heads tid / DH, tid / DH + GS, ...
  constexpr int GS = kAttnThreads / DH, NG = G / GS;
  static_assert(kAttnThreads % DH == 0 && G % GS == 0, "whole heads per round of threads");
  const int d = tid % DH, g0 = tid / DH;
  float o[NG], l[NG];
#pragma unroll
  for (int i = 0; i < NG; ++i) {
    const int g = g0 + i * GS;
    l[i] = (sums[0][g] + sums[1][g]) + (sums[2][g] + sums[3][g]);
    o[i] = 0.f;
#pragma unroll 8
    for (int j = 0; j < KPB; ++j) o[i] += accs[g][j * DH + d];
  }
  const auto leave = [&](int i, float v) { a.out[(int64_t)b * a.so_b + (int64_t)(h0 + g0 + i * GS) * a.so_h + d] = (uint16_t)E::bits(v); };
  if (ranges == 1) {
#pragma unroll
    for (int i = 0; i < NG; ++i) leave(i, l[i] > 0.f ? o[i] / l[i] : 0.f);
    return;
  }
  float* part_ws = a.ws_part + ((int64_t)(b * a.H + h0) * a.nsplit) * (DH + 2);      // [G][nsplit][DH + 2]
  const int64_t head_ws = (int64_t)a.nsplit * (DH + 2);
#pragma unroll
  for (int i = 0; i < NG; ++i) {
    float* mine = part_ws + (g0 + i * GS) * head_ws + (int64_t)s * (DH + 2);
    st_agent(mine + d, o[i]);
    if (d == 0) {
      float m = m_run[0];
#pragma unroll
      for (int g = 1; g < G; ++g) m = g == g0 + i * GS ? m_run[g] : m;
      st_agent(mine + DH, m);
      st_agent(mine + DH + 1, l[i]);
    }
  }
  wait_stores_acked();
  __syncthreads();
  int* count = &a.ws_count[b * a.H + h0];          // one arrival per split for the whole group
  if (tid == 0) {
    const int old = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last_flag = (old == ranges - 1);
  }
  __syncthreads();
  if (!last_flag) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  constexpr int SU = 8;
  float M[NG], num[NG], den[NG];
#pragma unroll
  for (int i = 0; i < NG; ++i) { M[i] = -INFINITY; num[i] = 0.f; den[i] = 0.f; }
  for (int i0 = 0; i0 < ranges; i0 += SU) {
    float mi[NG][SU];
#pragma unroll
    for (int i = 0; i < NG; ++i)
#pragma unroll
      for (int u = 0; u < SU; ++u) mi[i][u] = ld_agent(part_ws + (g0 + i * GS) * head_ws + (int64_t)min(i0 + u, ranges - 1) * (DH + 2) + DH);
#pragma unroll
    for (int i = 0; i < NG; ++i)
#pragma unroll
      for (int u = 0; u < SU; ++u) M[i] = fmaxf(M[i], mi[i][u]);
  }
  for (int i0 = 0; i0 < ranges; i0 += SU) {
    float mi[NG][SU], oi[NG][SU], li[NG][SU];
#pragma unroll
    for (int i = 0; i < NG; ++i)
#pragma unroll
      for (int u = 0; u < SU; ++u) {
        const float* pw = part_ws + (g0 + i * GS) * head_ws + (int64_t)min(i0 + u, ranges - 1) * (DH + 2);
        mi[i][u] = ld_agent(pw + DH);
        oi[i][u] = ld_agent(pw + d);
        li[i][u] = ld_agent(pw + DH + 1);
      }
#pragma unroll
    for (int i = 0; i < NG; ++i)
#pragma unroll
      for (int u = 0; u < SU; ++u) {
        const float w = (i0 + u >= ranges || mi[i][u] == -INFINITY) ? 0.f : __expf(mi[i][u] - M[i]);
        num[i] += w * oi[i][u];
        den[i] += w * li[i][u];
      }
  }
#pragma unroll
  for (int i = 0; i < NG; ++i) leave(i, den[i] > 0.f ? num[i] / den[i] : 0.f);
  if (tid == 0) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the appends of a call whose rows more than one workgroup reads
template <int DT>
__global__ __launch_bounds__(256) void kv_append_kernel(KvAppendArgs a) {
  const int half = a.Dh >> 1;
  const int total = a.B * a.Hk * half;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
    const int d = i % half, hk = (i / half) % a.Hk, b = i / (half * a.Hk);
    const int pos = a.seqlens[b];
    if (pos < 0 || pos >= a.S) continue;
    append_pair<DT>(a, half, b, hk, pos, d);
  }
}

size_t attn_decode_ws_floats(int B, int H, int nsplit, int Dh) { return (size_t)B * H * nsplit * (Dh + 2); }

template <int DT>
static void launch_attn_decode_t(const AttnDecodeArgs& a, int G, hipStream_t st) {
  dim3 grid(a.B * (a.H / G) * a.nsplit);
  if (G == 4 && a.Dh == 64) hipLaunchKernelGGL((attn_decode_gqa_kernel<DT, 64, 4, 4>), grid, dim3(kAttnThreads), 0, st, a);
  else if (G == 4) hipLaunchKernelGGL((attn_decode_gqa_kernel<DT, 128, 8, 4>), grid, dim3(kAttnThreads), 0, st, a);
  else if (G == 2) hipLaunchKernelGGL((attn_decode_gqa_kernel<DT, 128, 8, 2>), grid, dim3(kAttnThreads), 0, st, a);
  else if (a.Dh == 128) hipLaunchKernelGGL((attn_decode_kernel<DT, 128, 8>), grid, dim3(kAttnThreads), 0, st, a);
  else if (decode_one_pass(a.Dh, a.B, a.H, a.S, a.nsplit)) hipLaunchKernelGGL((attn_decode_kernel<DT, 64, 8, true>), grid, dim3(kAttnThreads), 0, st, a);
  else hipLaunchKernelGGL((attn_decode_kernel<DT, 64, 4>), grid, dim3(kAttnThreads), 0, st, a);
}

// true when the appended row of (b, hk) may be written by the launch that reads it, where one workgroup takes all query heads of the kv head: cache
// rows of different sequences and heads that do not overlap (sequences bound to one cache row see each other's new tokens, which takes a
// launch before this one)
static bool rows_apart(const AttnDecodeArgs& a) {
  return a.sc_h >= a.Dh && a.sc_s >= (a.Hk - 1) * a.sc_h + a.Dh && (a.B == 1 || a.sc_b >= a.S * a.sc_s);
}

int launch_attn_decode(const AttnDecodeArgs& args, hipStream_t st) {
  AttnDecodeArgs a = args;
  if (a.dt != 0 && a.dt != 1) { set_last_error("fsvd_attn_decode_densekv: dtype code %d (bf16 = 0 and fp16 = 1 are served)", a.dt); return kErrBadDtype; }
  if (a.B <= 0 || a.H <= 0 || a.Hk <= 0 || a.H % a.Hk != 0 || a.S <= 0 || a.nsplit <= 0) {
    set_last_error("fsvd_attn_decode_densekv: bad shape B=%d H=%d Hk=%d S=%d nsplit=%d", a.B, a.H, a.Hk, a.S, a.nsplit);
    return kErrBadShape;
  }
  if (a.Dh != 64 && a.Dh != 128) { set_last_error("fsvd_attn_decode_densekv: head_dim %d not in {64,128}", a.Dh); return kErrBadShape; }
  const int kpb = kAttnThreads / (a.Dh / 8);
  const int per = ((a.S + a.nsplit - 1) / a.nsplit + kpb - 1) / kpb * kpb;
  if (per > kMaxRowsPerRange) {
    set_last_error("fsvd_attn_decode_densekv: a cache of %d rows for %d key ranges (nsplit): at most %d rows a range", a.S, a.nsplit, kMaxRowsPerRange);
    return kErrBadShape;
  }
  if ((a.sc_s % 8) || (a.sc_h % 8) || (a.sc_b % 8) || (reinterpret_cast<uintptr_t>(a.k_cache) & 15) ||
      (reinterpret_cast<uintptr_t>(a.v_cache) & 15)) {
    set_last_error("fsvd_attn_decode_densekv: cache strides/pointers must be 16-byte aligned");
    return kErrBadAlign;
  }
  if (a.nsplit > 1 && (!a.ws_part || !a.ws_count)) { set_last_error("fsvd_attn_decode_densekv: workspace missing"); return kErrWorkspace; }
  const bool own = a.k_new != nullptr && rows_apart(a);
  const int G = decode_group(a.Dh, a.B, a.H, a.Hk, a.S, a.nsplit, own);
  a.plan = decode_plan(a.Dh, G, a.B, a.H, a.Hk, a.nsplit);
  if (a.k_new && !(own && a.H / a.Hk == G)) {
    const KvAppendArgs ka{a.k_new, a.v_new, a.sk_b, a.sk_h, a.sv_b, a.sv_h, const_cast<uint16_t*>(a.k_cache), const_cast<uint16_t*>(a.v_cache),
                          a.sc_b, a.sc_s, a.sc_h, a.seqlens, a.cos, a.sin, a.rope_len, a.B, a.Hk, a.Dh, a.S, a.dt};
    const int rc = launch_kv_append(ka, st);
    if (rc != kOk) return rc;
    a.k_new = nullptr;
  }
  if (a.dt == 1) launch_attn_decode_t<1>(a, G, st);
  else launch_attn_decode_t<0>(a, G, st);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_last_error("fsvd_attn_decode_densekv: launch failed: %s", hipGetErrorString(e)); return kErrLaunch; }
  return kOk;
}

int launch_kv_append(const KvAppendArgs& a, hipStream_t st) {
  if (a.B <= 0 || a.Hk <= 0 || a.Dh <= 0 || (a.Dh & 1) || a.S <= 0) { set_last_error("fsvd_kv_append: bad shape"); return kErrBadShape; }
  const int total = a.B * a.Hk * (a.Dh / 2);
  if (a.dt != 0 && a.dt != 1) { set_last_error("fsvd_kv_append: dtype code %d (bf16 = 0 and fp16 = 1 are served)", a.dt); return kErrBadDtype; }
  if (a.dt == 1) hipLaunchKernelGGL(kv_append_kernel<1>, dim3((total + 255) / 256), dim3(256), 0, st, a);
  else hipLaunchKernelGGL(kv_append_kernel<0>, dim3((total + 255) / 256), dim3(256), 0, st, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_last_error("fsvd_kv_append: launch failed: %s", hipGetErrorString(e)); return kErrLaunch; }
  return kOk;
}

}  // namespace fsvd
