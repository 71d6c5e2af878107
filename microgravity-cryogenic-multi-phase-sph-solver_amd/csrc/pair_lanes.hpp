// Shared by the neighbour passes: several lanes per target particle, prefetched
// loads, spans of particles by XCD.
#pragma once

#include <type_traits>

#include "kernels.hpp"

namespace cryo {
namespace {

constexpr int kBlock = 256;
__device__ inline int gtid() { return static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x); }
inline int blocks_for(long long n) { return static_cast<int>((n + kBlock - 1) / kBlock); }

// Max of non-negative floats (NaN ignored, as `v > acc ? v : acc` does).
__device__ inline float wave_max(float v) {
  for (int off = 32; off > 0; off >>= 1) {
    const float o = __shfl_down(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}
__device__ inline void atomic_max_nonneg(unsigned* addr, float v) {
  if (v > 0.0f) atomicMax(addr, __float_as_uint(v));
}

// pow for positive float arguments: evaluated in double and rounded once.
__device__ inline float powf_cr(float x, float y) { return static_cast<float>(pow(static_cast<double>(x), static_cast<double>(y))); }

// G neighbouring lanes share one target particle: lane k of the group takes
// neighbours k, k + G, ... of the particle's list, evaluates its pair, and the
// pairs' terms are then added in list order by every lane of the group, each
// term read from the lane that holds it (a quad broadcast in the add's own
// operand).  The sums therefore see the reference's order, whatever G is.
template <int G>
struct Lanes {
  static_assert(G == 2 || G == 4 || G == 16, "a quad's parts, or a row of 16 lanes");
  // every lane of the group gets lane k's v
  template <int K>
  __device__ static inline float from(float v) {
    constexpr int b = G == 2 ? 2 + K : K;
    constexpr int ctrl = G == 16 ? 0x150 + K : K | (K << 2) | (b << 4) | (b << 6);  // row_newbcast or quad_perm
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xf, 0xf, true));
  }
  template <int K>
  __device__ static inline V3 from(V3 v) {
    return V3{from<K>(v.x), from<K>(v.y), from<K>(v.z)};
  }
  // the wave's lanes that are lane k of their group
  static constexpr unsigned long long mask(int k) {
    unsigned long long m = 0;
    for (int l = k; l < 64; l += G) m |= 1ull << l;
    return m;
  }
};
template <int N, class F>
__device__ inline void unrolled(F&& f) {
  if constexpr (N > 0) {
    unrolled<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// A value that is the same in every lane, kept in a scalar register.
__device__ inline float uniform(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// v moved to a register of its own, here: the wait for a load into v falls at
// this point, and v's register is free for the next load.  (Rotating a
// prefetched value by assignment lets the compiler place the move, and with
// it the wait, right behind the load.)
__device__ inline float take(float v) {
  float r;
  asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}
__device__ inline int take(int v) {
  int r;
  asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}
__device__ inline float4 take(float4 v) { return make_float4(take(v.x), take(v.y), take(v.z), take(v.w)); }

// Block b of an nblocks grid -> the span of particles it runs.  The hardware
// deals workgroups round-robin to the 8 XCDs (XCD b % 8); within each group of
// 8 x kSpanChunk blocks, XCD x runs kSpanChunk consecutive spans, so that
// neighbouring spans, which read the same records, meet in one L2.  The last,
// partial group keeps the identity.  A bijection of [0, nblocks).
constexpr int kSpanChunk = 16;
__device__ inline int xcd_span(int b, int nblocks) {
  constexpr int span = 8 * kSpanChunk;
  if (b >= nblocks / span * span) return b;
  return b / span * span + (b % 8) * kSpanChunk + (b / 8) % kSpanChunk;
}

// Orders this wave's LDS writes before its later reads (the hardware does; this
// keeps the compiler from moving them).
__device__ inline void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// One block's particles [base, base + span), span <= kBlock: select(i) says
// whether particle i takes part (and writes what the others get); the selected
// ones, in order, go to groups of G lanes, body(i, sub) once per lane of a
// group.  Every thread of the block calls it.
template <int G, class Select, class Body>
__device__ inline void for_each_group(int base, int span, int n, Select&& select, Body&& body) {
  __shared__ int s_work[kBlock], s_tot[kBlock / 64];
  const int t = static_cast<int>(threadIdx.x), lane = t & 63, wave = t >> 6;
  const bool keep = t < span && base + t < n && select(base + t);
  const unsigned long long kept = __ballot(keep);
  if (lane == 0) s_tot[wave] = __popcll(kept);
  __syncthreads();
  int first = 0, total = 0;
  for (int w = 0; w < kBlock / 64; ++w) {
    const int c = s_tot[w];
    first += w < wave ? c : 0;
    total += c;
  }
  if (keep) s_work[first + __popcll(kept & ((1ull << lane) - 1ull))] = base + t;
  __syncthreads();
  for (int slot = t / G; slot < total; slot += kBlock / G) body(s_work[slot], t % G);
}

// Sums over particle i's neighbours by its group of G lanes: eval(j, t) sets
// the terms t[0..N) of neighbour j (they come in as zeros), which are added to
// acc in list order.  Without a complete list every lane walks the 27 cells.
template <int G, int N, bool KS, class Eval>
__device__ inline void lane_sums(const NbrList& L, const GridDev& g, int i, V3 xi, int sub, Acc<KS> (&acc)[N],
                                 Eval&& eval) {
  const int c = L.valid ? L.count[i] : -1;
  if (c < 0) {
    for_each_nbr(g, xi, [&](int j) {
      float t[N] = {};
      eval(j, t);
#pragma unroll
      for (int q = 0; q < N; ++q) acc[q] += t[q];
    });
    return;
  }
  const int* lp = reinterpret_cast<const int*>(list_chunks(L, i));
  int jn = sub < c ? lp[(sub >> 2) * (4 * kListGroup) + (sub & 3)] : -1;
  for (int e = sub; e - sub < c; e += G) {
    const int j = take(jn);
    jn = e + G < c ? lp[((e + G) >> 2) * (4 * kListGroup) + ((e + G) & 3)] : -1;
    float t[N] = {};
    if (j >= 0) eval(j, t);
    unrolled<G>([&](auto kc) {
#pragma unroll
      for (int q = 0; q < N; ++q) acc[q] += Lanes<G>::template from<decltype(kc)::value>(t[q]);
    });
  }
}

}  // namespace
}  // namespace cryo
