// The few words of state between two decoded tokens: the greedy token of every row and its next position, and the state that a
// caller sets before a step, one launch each instead of a chain of library launches.
//   greedy token, one sequence of 32000 logits, on every token of the graph engine: the library's argmax took 13.0 us, the copy of its
//     result and the position increment 6 with their gaps; this takes 3.8, bound by the one compute unit that reads the row.
//   state, once per prompt in a generation: three 4-byte copies of 3 to 6 us each in front of the resident step, two in front of a
//     graph -> one launch.  The steps advance their own state, so a generated token gains nothing from it; a program that sets the
//     state before every token of the resident step saves 46 us on each.
#include "common.hpp"
#include "../../include/flashsvd_hip.h"

namespace fsvd {

constexpr int kPickThreads = 1024, kPickLoads = 4;

// 16-bit patterns as integers in the order of their values: NaN above everything, the two zeros equal
template <int DT>
__device__ __forceinline__ uint32_t order_key(uint32_t p) {
  const uint32_t mag = p & 0x7fffu;
  if (mag > (DT == 1 ? 0x7c00u : 0x7f80u)) return 0x10000u;
  if (mag == 0) return 0x8000u;
  return (p & 0x8000u) ? 0xffffu - p : p | 0x8000u;
}

// two 16-bit patterns as unsigned 16-bit integers in the order of their values (a NaN above everything of its sign, -0 next below +0)
typedef short i16x2_t __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2_t order_pair(uint32_t w) {
  const i16x2_t p = __builtin_bit_cast(i16x2_t, w);
  return __builtin_bit_cast(u16x2_t, (i16x2_t)(p ^ ((p >> 15) | (short)0x8000)));
}

// Rows of at most two 16-byte pieces per thread: value and index together, element by element, in one reduction.  What a launch takes is its two
// round trips and the reductions, and the kernel below has three of those: us per launch in a graph there / here, 1000 logits of 1 / 64 rows 3.5 / 2.6, 4.0 /
// 3.0, 8192 3.7 / 3.1, 4.1 / 3.6, 14336 3.7 / 3.6, 4.2 / 4.1; 16384 3.7 / 3.9, 4.2 / 4.4, hence the line.
constexpr int kShortLoads = 2, kShortRow = 14336;
static_assert(kShortRow <= kPickThreads * kShortLoads * 8, "two pieces per thread");
template <int DT>
__global__ __launch_bounds__(kPickThreads) void greedy_short_kernel(const uint16_t* __restrict__ logits, int64_t ld, int64_t* __restrict__ tokens,
                                                                   int64_t ldt, int32_t* __restrict__ positions, int V) {
  const uint16_t* row = logits + (int64_t)blockIdx.x * ld;
  const int tid = threadIdx.x, pieces = V >> 3;
  uint32_t best = 0, at = 0x7fffffffu;
  const auto take = [&](uint32_t p, uint32_t i) {
    const uint32_t k = order_key<DT>(p);
    if (k > best) { best = k; at = i; }                // a thread meets its elements in ascending order
  };
  u32x4_t v[kShortLoads];
#pragma unroll
  for (int j = 0; j < kShortLoads; ++j)
    if (j * kPickThreads + tid < pieces) v[j] = *reinterpret_cast<const u32x4_any_t*>(row + (j * kPickThreads + tid) * 8);
#pragma unroll
  for (int j = 0; j < kShortLoads; ++j) {
    const int c = j * kPickThreads + tid;
    if (c >= pieces) break;
    const uint32_t w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
    for (int e = 0; e < 8; ++e) take((w[e >> 1] >> (16 * (e & 1))) & 0xffffu, c * 8 + e);
  }
  if (pieces * 8 + tid < V) take(row[pieces * 8 + tid], pieces * 8 + tid);
  unsigned long long m = ((unsigned long long)best << 32) | (0xffffffffu - at);
#pragma unroll
  for (int o = 32; o; o >>= 1) {
    const unsigned long long other = __shfl_xor(m, o);
    m = other > m ? other : m;
  }
  __shared__ unsigned long long red[kPickThreads / kWave];
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int i = 1; i < kPickThreads / kWave; ++i) m = red[i] > m ? red[i] : m;
    tokens[(int64_t)blockIdx.x * ldt] = (int64_t)(0xffffffffu - (uint32_t)m);
    if (positions) positions[blockIdx.x] += 1;
  }
}

// One workgroup per row: the row is requested in rounds of four 16-byte pieces per thread (32768 elements), so what it takes is
// one round trip per round and the 60 GB/s of one compute unit.  Beside that every instruction per element shows, 32 of them in a thread: a
// first pass takes the maximum alone, two elements to an instruction; then the threads that hold it look for it in the round where they met
// it.  us per launch in a graph, value and index carried along element by element -> this: 32000 logits of 1 / 16 / 64 rows 5.3 -> 3.8, 5.9 -> 4.2,
// 6.1 -> 4.4, 128256 of 1 / 16 rows 14.7 -> 6.0, 15.2 -> 6.5.  Ties go to the lowest index and NaN counts as the largest value, as torch.argmax
// has it: a row with a NaN (its largest magnitude tells), or whose largest value is a zero of either sign, is looked through element by element (32000 zeros 6.4).
template <int DT>
__global__ __launch_bounds__(kPickThreads) void greedy_token_kernel(const uint16_t* __restrict__ logits, int64_t ld, int64_t* __restrict__ tokens,
                                                                   int64_t ldt, int32_t* __restrict__ positions, int V) {
  const uint16_t* row = logits + (int64_t)blockIdx.x * ld;
  const int tid = threadIdx.x, pieces = V >> 3;
  __shared__ uint32_t top[kPickThreads / kWave], far[kPickThreads / kWave], first[kPickThreads / kWave];
  const auto fetch = [&](int c0, u32x4_t (&v)[kPickLoads]) {
#pragma unroll
    for (int j = 0; j < kPickLoads; ++j) v[j] = *reinterpret_cast<const u32x4_any_t*>(row + (int64_t)min(c0 + j * kPickThreads + tid, pieces - 1) * 8);
  };
  u32x4_t v[kPickLoads];
  constexpr int kTail = -1;
  uint32_t best = 0, mag = 0;                          // the largest of this thread and the largest magnitude
  int where = 0;                                       // the first round with the largest
  for (int c0 = 0; c0 < pieces; c0 += kPickThreads * kPickLoads) {
    fetch(c0, v);
    u16x2_t most = {0, 0}, wide = {0, 0};
#pragma unroll
    for (int j = 0; j < kPickLoads; ++j) {             // pieces past the end are the last one once more
      const uint32_t w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        most = __builtin_elementwise_max(most, order_pair(w[e]));
        wide = __builtin_elementwise_max(wide, __builtin_bit_cast(u16x2_t, w[e] & 0x7fff7fffu));
      }
    }
    const uint32_t k = max((uint32_t)most.x, (uint32_t)most.y);
    if (k > best) { best = k; where = c0; }
    mag = max(mag, max((uint32_t)wide.x, (uint32_t)wide.y));
  }
  const int t = pieces * 8 + tid;                      // at most seven elements behind the last piece
  const uint32_t tail = t < V ? row[t] : 0xffffu;
  if (t < V) {
    const uint32_t k = order_pair(tail).x;
    if (k > best) { best = k; where = kTail; }
    mag = max(mag, tail & 0x7fffu);
  }
  const auto all_max = [&](uint32_t x, uint32_t* red) {
#pragma unroll
    for (int o = 32; o; o >>= 1) x = max(x, (uint32_t)__shfl_xor((int)x, o));
    if ((tid & 63) == 0) red[tid >> 6] = x;
  };
  all_max(best, top);
  all_max(mag, far);
  __syncthreads();
  uint32_t highest = 0, widest = 0;
#pragma unroll
  for (int i = 0; i < kPickThreads / kWave; ++i) { highest = max(highest, top[i]); widest = max(widest, far[i]); }
  // the lowest index that holds the largest value
  uint32_t at = 0xffffffffu;
  const auto look = [&](int c0, auto hit) {
#pragma unroll
    for (int j = 0; j < kPickLoads; ++j) {
      const uint32_t w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
      const int c = c0 + j * kPickThreads + tid;
      if (c >= pieces) break;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (hit((w[e >> 1] >> (16 * (e & 1))) & 0xffffu)) at = min(at, (uint32_t)(c * 8 + e));
    }
  };
  constexpr int kRound = kPickThreads * kPickLoads;
  if (widest > (DT == 1 ? 0x7c00u : 0x7f80u) || highest == 0x8000u) {      // a NaN, or zero, which -0 equals
    const uint32_t least = highest == 0x8000u && widest <= (DT == 1 ? 0x7c00u : 0x7f80u) ? 0x8000u : 0x10000u;
    const auto hit = [&](uint32_t p) { return order_key<DT>(p) >= least; };
    for (int c0 = 0; c0 < pieces; c0 += kRound) {
      fetch(c0, v);
      look(c0, hit);
    }
    if (t < V && hit(tail)) at = min(at, (uint32_t)t);
  } else if (best == highest) {
    if (where == kTail) {
      at = (uint32_t)t;
    } else {
      if (where + kRound < pieces) fetch(where, v);    // not the round that is still in registers
      look(where, [&](uint32_t p) { return (uint32_t)order_pair(p).x == highest; });
    }
  }
#pragma unroll
  for (int o = 32; o; o >>= 1) at = min(at, (uint32_t)__shfl_xor((int)at, o));
  if ((tid & 63) == 0) first[tid >> 6] = at;
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int i = 1; i < kPickThreads / kWave; ++i) at = min(at, first[i]);
    tokens[(int64_t)blockIdx.x * ldt] = (int64_t)at;
    if (positions) positions[blockIdx.x] += 1;
  }
}

__global__ void step_state_kernel(fsvd_step_state* st, int64_t token, int32_t pos) {
  st->pos = pos;
  st->step = 0;
  st->token = token;
}

__global__ void token_rows_kernel(int64_t* tokens, const int64_t* src, int32_t* positions, int32_t pos, int B) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  tokens[b] = src[b];
  positions[b] = pos;
}

static int launched(const char* fn) {
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return kOk;
  set_last_error("%s: launch failed: %s", fn, hipGetErrorString(e));
  return kErrLaunch;
}

}  // namespace fsvd

using namespace fsvd;

extern "C" {

int fsvd_greedy_token(const void* logits, int64_t ld, int64_t* tokens, int64_t ldt, int32_t* positions, int B, int V, int dtype, void* stream) {
  const char* fn = "fsvd_greedy_token";
  if (logits == nullptr || tokens == nullptr) { set_last_error("%s: argument %s is NULL", fn, logits == nullptr ? "logits" : "tokens"); return kErrNullPtr; }
  if (B <= 0 || V <= 0) { set_last_error("%s: empty shape (B = %d, V = %d)", fn, B, V); return kErrBadShape; }
  if (dtype != 0 && dtype != 1) { set_last_error("%s: dtype code %d (bf16 = 0 and fp16 = 1 are served)", fn, dtype); return kErrBadDtype; }
  if ((reinterpret_cast<uintptr_t>(logits) & 1) != 0) { set_last_error("%s: logits must be 2-byte aligned", fn); return kErrBadAlign; }
  const auto* x = static_cast<const uint16_t*>(logits);
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (V <= kShortRow) {
    if (dtype == 1) hipLaunchKernelGGL(greedy_short_kernel<1>, dim3(B), dim3(kPickThreads), 0, st, x, ld, tokens, ldt, positions, V);
    else hipLaunchKernelGGL(greedy_short_kernel<0>, dim3(B), dim3(kPickThreads), 0, st, x, ld, tokens, ldt, positions, V);
  } else if (dtype == 1) hipLaunchKernelGGL(greedy_token_kernel<1>, dim3(B), dim3(kPickThreads), 0, st, x, ld, tokens, ldt, positions, V);
  else hipLaunchKernelGGL(greedy_token_kernel<0>, dim3(B), dim3(kPickThreads), 0, st, x, ld, tokens, ldt, positions, V);
  return launched(fn);
}

int fsvd_decode_step_set_state(fsvd_step_state* state, int64_t token, int32_t position, void* stream) {
  const char* fn = "fsvd_decode_step_set_state";
  if (state == nullptr) { set_last_error("%s: argument state is NULL", fn); return kErrNullPtr; }
  hipLaunchKernelGGL(step_state_kernel, dim3(1), dim3(1), 0, static_cast<hipStream_t>(stream), state, token, position);
  return launched(fn);
}

int fsvd_set_token_rows(int64_t* tokens, const int64_t* src, int32_t* positions, int32_t position, int B, void* stream) {
  const char* fn = "fsvd_set_token_rows";
  if (tokens == nullptr || src == nullptr || positions == nullptr) { set_last_error("%s: a buffer is NULL", fn); return kErrNullPtr; }
  if (B <= 0) { set_last_error("%s: empty shape (B = %d)", fn, B); return kErrBadShape; }
  hipLaunchKernelGGL(token_rows_kernel, dim3((B + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream), tokens, src, positions, position, B);
  return launched(fn);
}

}  // extern "C"
