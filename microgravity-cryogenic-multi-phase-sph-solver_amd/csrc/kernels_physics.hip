// Neighbour-loop physics on gfx950.
//
// The reference runs one kernel per operator (evaluate_rates,
// sph_solver.cu:449-480).  Here operators whose inputs are ready at the same
// point share one neighbour sweep:
//   k_density    density summation + EOS          (SPH_kernels.cu:6-34, navier_stokes.cu:5-14)
//   k_wall_bc    Adami wall extrapolation          (navier_stokes.cu:16-69)
//   k_interface  colour gradient, alpha, wall/heat weights, contact angle, SPS,
//                pointwise CSF normals             (surface_tension.cu:5-118, navier_stokes.cu:71-119)
//   k_forces     everything else of the rates (kernels_forces.hpp)
// Every accumulator adds its neighbours in the reference order (ascending
// sorted index), with the reference's per-pair expressions, so each field is
// the same float the reference computes (given equal inputs).
#include <algorithm>
#include <stdexcept>

#include "pair_lanes.hpp"

namespace cryo {

namespace {

// Deterministic FP64 block sum: fixed shuffle tree per wave, waves in order.
__device__ inline void block_sum_store(double v, double* out) {
  __shared__ double wsum[kBlock / 64];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) wsum[wave] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0;
    for (int w = 0; w < kBlock / 64; ++w) s += wsum[w];
    *out = s;
  }
}

// W at squared distance r2 (below r2_fast it is its value at 0 to the last bit).
__device__ inline float kernel_at(const SimParams& P, float r2) {
  return kW(P.kernel, P.fast ? sqrt_rn(r2 < P.r2_fast ? P.r2_fast : r2) : sqrtf(r2));
}

// Density, pressure and neighbour record of particle i from its kernel sum and
// squared nearest distance.
template <bool KS>
__device__ inline void density_finish(const PV& pv, const SimParams& P, int i, const Acc<KS>& sum, float r2min) {
  const uint8_t ph = pv.s.phase[i];
  const V3 xi = ld3(pv.s.x[i]);
  if (!is_fluid(ph)) {
    pv.t.sigma[i] = 1.0f / P.vol0;
    pv.t.rmin[i] = P.kernel.support;
    if (ph != kWall) {  // dead, not yet dropped: what the last evaluation gave it, at its present phase and velocity
      const float4 v = pv.s.v[i];
      PairRec& rec = pv.t.rec[i];
      rec.x = make_float4(xi.x, xi.y, xi.z, __int_as_float(ph));
      rec.v = make_float4(v.x, v.y, v.z, rec.v.w);
      rec.t = st3(ld3(pv.s.vt[i]));
    }
    return;
  }
  pv.t.sigma[i] = float(sum);
  pv.t.rmin[i] = sqrtf(r2min);
  float rho = pv.s.rho[i];
  const float mi = pv.s.m[i];
  const float Ti = pv.s.T[i];
  float p;
  if constexpr (KS) {
    // precision form: the summation density in double, the EOS on it
    double rho_d = rho;
    if (P.density_mode == 0) {
      rho_d = static_cast<double>(ph == kLiquid ? pv.s.m0[i] : mi) * (static_cast<double>(sum.s) + sum.c);
      rho = static_cast<float>(rho_d);
      pv.s.rho[i] = rho;
    }
    p = eos_pressure_hp(P, ph, rho_d, Ti);
  } else {
    if (P.density_mode == 0) {
      rho = (ph == kLiquid ? pv.s.m0[i] : mi) * float(sum);
      pv.s.rho[i] = rho;
    }
    p = eos_pressure(P, ph, rho, Ti);
  }
  pv.t.p[i] = p;
  const float4 q = make_float4(p, mi, rho, Ti);
  const float V = mi / rho;
  pv.t.vol[i] = V;
  const float4 v = pv.s.v[i], vt = pv.s.vt[i];
  pv.t.rec[i] = PairRec{make_float4(xi.x, xi.y, xi.z, __int_as_float(ph)), q, make_float4(v.x, v.y, v.z, V),
                        make_float4(vt.x, vt.y, vt.z, P.tvf ? 1.0f / float(sum) : 0.0f)};
}

// ------------------------------------------------------- density + EOS
// Also builds the step's neighbour lists from the same (cell-culled) sweep.
// A row of 16 lanes takes one particle: its lanes 0..8 look the nine cell rows
// up side by side, then the lanes test 16 candidates at a time; the hits, in
// candidate order, go to the list and their squared distances to LDS, from
// where 16 kernel values at a time are evaluated and added in order.  (One
// thread per particle ran a chain of about 350 candidate tests, and the kernel
// evaluation for every one that any lane of the wave hit: 156 us at any size
// up to 100 k particles; now 28 us at 26 k.)  A block takes 16 consecutive
// particles and writes their results coalesced.
constexpr int kDensLanes = 16;
constexpr int kDensRing = 128;  // hits of one particle waiting for their kernel values
template <bool KS>
__global__ __launch_bounds__(kBlock) void k_density(PV pv, GridDev g, SimParams P, NbrList L, Count nc) {
  constexpr int kGroups = kBlock / kDensLanes, kSpan = kGroups;
  using Ln = Lanes<kDensLanes>;
  __shared__ int2 s_row[kGroups][9];           // one past the row's last candidate number; sorted index - number
  __shared__ float s_r2[kGroups][kDensRing];
  __shared__ float s_sum[kSpan], s_low[kSpan], s_min[kSpan];
  __shared__ int s_count[kSpan];
  const int n = nc.get();
  const int base = xcd_span(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x)) * kSpan;
  if (base >= n) return;  // uniform over the block
  const int grp = static_cast<int>(threadIdx.x) / kDensLanes, l = threadIdx.x % kDensLanes;
  const int lane = threadIdx.x & 63;
  const int row0 = lane & ~(kDensLanes - 1);
  const float4* __restrict__ xs = pv.s.x;
  const int me = base + grp;
  const bool here = me < n;
  const uint8_t ph = here ? pv.s.phase[me] : kDead;
  const bool fluid = is_fluid(ph);
  const V3 xi = here ? ld3(xs[me]) : V3{0, 0, 0};
  V3 li{0, 0, 0};
  if (KS && fluid) li = ld3(pv.s.xlo[me]);
  // the nine rows of the 27 cells (for_each_cand), one per lane
  const float ux = (xi.x - g.ox) * g.inv_cell, uy = (xi.y - g.oy) * g.inv_cell, uz = (xi.z - g.oz) * g.inv_cell;
  const int cx = clampv(static_cast<int>(floorf(ux)), 0, g.nx - 1);
  const int cy = clampv(static_cast<int>(floorf(uy)), 0, g.ny - 1);
  const int cz = clampv(static_cast<int>(floorf(uz)), 0, g.nz - 1);
  const int dz = l / 3 - 1, dy = l % 3 - 1;
  const int z = cz + dz, y = cy + dy;
  int first = 0, len = 0;
  bool near_fluid = false;
  if (here && ph != kDead && l < 9 && z >= 0 && z < g.nz && y >= 0 && y < g.ny) {
    const int row = (z * g.ny + y) * g.nx;
    const float fx = ux - static_cast<float>(cx), fy = uy - static_cast<float>(cy), fz = uz - static_cast<float>(cz);
    const float rc = P.kernel.support * g.inv_cell + g.cull_pad;
    const float rr = rc * rc;
    const float gz = dz < 0 ? fz : (dz > 0 ? 1.0f - fz : 0.0f);
    const float gy = dy < 0 ? fy : (dy > 0 ? 1.0f - fy : 0.0f);
    const float gyz = gy * gy + gz * gz;
    if (!(gyz >= rr)) {
      const int x0 = (cx > 0 && gyz + fx * fx < rr) ? cx - 1 : cx;
      const int x1 = (cx < g.nx - 1 && gyz + (1.0f - fx) * (1.0f - fx) < rr) ? cx + 1 : cx;
      first = g.off[row + x0];
      len = g.off[row + x1 + 1] - first;
    }
    if (!fluid) {
      const int x0 = cx > 0 ? cx - 1 : 0, x1 = cx < g.nx - 1 ? cx + 1 : cx;
      int any = 0;
      for (int x = x0; x <= x1; ++x) any |= g.flags[row + x];
      near_fluid = (any & kCellFluid) != 0;
    }
  }
  // wall targets only ever need their fluid neighbours: none without a fluid
  // particle in the 27 cells
  const unsigned rows_fluid = static_cast<unsigned>(__ballot(near_fluid) >> row0) & 0xffffu;
  if (!fluid && rows_fluid == 0) len = 0;
  int end = len;
#pragma unroll
  for (int off = 1; off < kDensLanes; off <<= 1) {
    const int o = __shfl_up(end, off, kDensLanes);
    if (l >= off) end += o;
  }
  if (l < 9) s_row[grp][l] = make_int2(end, first - (end - len));
  const int total = __shfl(end, kDensLanes - 1, kDensLanes);
  wave_lds_fence();
  Acc<KS> sum;
  float r2min = P.support2;
  int c = 0, done = 0;
  int* out = reinterpret_cast<int*>(list_chunks(L, here ? me : 0));
  // adds the kernel values of hits [done, done + 16) below c
  auto drain = [&]() {
    const int k = done + l;
    const float r2 = s_r2[grp][k & (kDensRing - 1)];
    float w = 0.0f;
    if (k < c) w = kernel_at(P, r2);
    unrolled<kDensLanes>([&](auto kc) { sum += Ln::template from<decltype(kc)::value>(w); });
    done += kDensLanes;
  };
  int2 row = s_row[grp][0];
  int r = 0;
  auto index = [&](int v) {  // sorted index of candidate v; the particle itself past the end
    if (v >= total) return here ? me : 0;
    while (v >= row.x) row = s_row[grp][++r];
    return v + row.y;
  };
  int j = index(l);
  float4 x = xs[j];
  uint8_t q = kLiquid;
  if (!fluid) q = pv.s.phase[j];
  for (int v = l; __any(v - l < total); v += kDensLanes) {
    const float4 xj = take(x);
    const int jc = j;
    const bool usable = v < total && (fluid || is_fluid(q));
    if (v - l + kDensLanes < total) {
      j = index(v + kDensLanes);
      x = xs[j];
      if (!fluid) q = pv.s.phase[j];
    }
    // neighbourhood by the float positions (the lists of every later pass);
    // in the precision form the kernel takes the double-float distance
    const float r2h = norm2(xi - ld3(xj));
    const bool hit = usable && !(r2h >= P.support2);
    const unsigned hits = static_cast<unsigned>(__ballot(hit) >> row0) & 0xffffu;
    if (hit) {
      const int e = c + __popc(hits & ((1u << l) - 1u));
      if (e < L.K) out[(e >> 2) * (4 * kListGroup) + (e & 3)] = jc;
      if (fluid) {
        const float r2 = KS ? norm2(pos_diff<KS>(xi, li, ld3(xj), pv.s.xlo, jc)) : r2h;
        if (jc != me && r2 < r2min) r2min = r2;
        s_r2[grp][e & (kDensRing - 1)] = r2;
      }
    }
    c += __popc(hits);
    if (__any(fluid && c - done > kDensRing - kDensLanes)) {
      wave_lds_fence();
      if (fluid)
        while (c - done >= kDensLanes) drain();
    }
  }
  wave_lds_fence();
  if (fluid)
    while (done < c) drain();
  for (int off = kDensLanes / 2; off > 0; off >>= 1) {
    const float o = __shfl_xor(r2min, off, kDensLanes);
    r2min = o < r2min ? o : r2min;
  }
  if (l == 0) {
    if constexpr (KS) {
      s_sum[grp] = sum.s;
      s_low[grp] = sum.c;
    } else {
      s_sum[grp] = sum;
    }
    s_min[grp] = r2min;
    s_count[grp] = c <= L.K ? c : -1;
  }
  __syncthreads();
  const int slot = threadIdx.x;
  const int i = base + slot;
  if (slot >= kSpan || i >= n) return;
  L.count[i] = s_count[slot];
  Acc<KS> whole;
  whole.s = s_sum[slot];
  if constexpr (KS) whole.c = s_low[slot];
  density_finish<KS>(pv, P, i, whole, s_min[slot]);
}

// One thread per particle: what very large sets take (from kDensWide on, where
// every SIMD is full either way and the shorter chains of the row of lanes
// above no longer pay for its bookkeeping).  us with the row / with one thread:
//   two-phase sphere  188 k 131 / 184, 420 k 273 / 287, 550 k 361 / 373, 700 k 455 / 444, 1.2 M 787 / 693
//   precise  188 k 183 / 256, 420 k 387 / 467, 550 k 501 / 548, 700 k 633 / 628, 1.2 M 1099 / 1019
//   column  297 k 131 / 176, 550 k 236 / 238, 696 k 311 / 301, 1 M 451 / 407
constexpr int kDensWide = 600000;
template <bool KS>
__global__ __launch_bounds__(kBlock) void k_density_wide(PV pv, GridDev g, SimParams P, NbrList L, Count nc) {
  const int n = nc.get();
  const int i = gtid();
  if (i >= n) return;
  const uint8_t ph = pv.s.phase[i];
  const V3 xi = ld3(pv.s.x[i]);
  ListWriter lw(L, i);
  Acc<KS> sum;
  float r2min = P.support2;
  if (!is_fluid(ph)) {
    // wall targets only ever need their fluid neighbours: none without a fluid
    // particle in the 27 cells
    if (ph == kWall && cells_any(g, xi, kCellFluid)) {
      for_each_cand_xph(g, xi, P.kernel.support, pv.s.x, pv.s.phase, [&](int j, float4 xj, uint8_t phj) {
        if (norm2(xi - ld3(xj)) >= P.support2) return;
        if (!is_fluid(phj)) return;
        lw.push(j);
      });
    }
  } else {
    const V3 li = pos_lo<KS>(pv.s.xlo, i);
    for_each_cand_x(g, xi, P.kernel.support, pv.s.x, [&](int j, float4 xj) {
      // neighbourhood by the float positions (the lists of every later pass);
      // in the precision form the kernel takes the double-float distance
      const float r2h = norm2(xi - ld3(xj));
      if (r2h >= P.support2) return;
      const float r2 = KS ? norm2(pos_diff<KS>(xi, li, ld3(xj), pv.s.xlo, j)) : r2h;
      sum += kernel_at(P, r2);
      if (j != i && r2 < r2min) r2min = r2;
      lw.push(j);
    });
  }
  L.count[i] = lw.finish();
  density_finish<KS>(pv, P, i, sum, r2min);
}

// SPH_kernels.cu:36-54 (start-up only).
template <bool KS>
__global__ __launch_bounds__(kBlock) void k_normalize_masses(PV pv, GridDev g, SimParams P, int n) {
  const int i = gtid();
  if (i >= n) return;
  if (!is_fluid(pv.s.phase[i])) return;
  const V3 xi = ld3(pv.s.x[i]);
  const V3 li = pos_lo<KS>(pv.s.xlo, i);
  // the same sum the density pass forms (compensated in the precision form),
  // so that the start state sits at rho0 in either form
  Acc<KS> acc;
  for_each_nbr(g, xi, [&](int j) {
    const V3 xj = ld3(pv.s.x[j]);
    if (norm2(xi - xj) >= P.support2) return;
    acc += kW(P.kernel, sqrtf(KS ? norm2(pos_diff<KS>(xi, li, xj, pv.s.xlo, j)) : norm2(xi - xj)));
  });
  const float sum = float(acc);
  if (sum > 0.0f) {
    const float m = pv.s.rho[i] / sum;
    pv.s.m[i] = m;
    pv.s.m0[i] = m;
  }
}

// --------------------------------------------------------------- wall BC
template <bool KS>
__global__ __launch_bounds__(kBlock) void k_wall_bc(PV pv, GridDev g, SimParams P, NbrList L, const DevState* st,
                                                   Count nc) {
  const int n = nc.get();
  const int i = gtid();
  if (i >= n) return;
  if (pv.s.phase[i] != kWall) return;
  const V3 grav = st->gravity;
  const V3 xi = ld3(pv.s.x[i]);
  const V3 li = pos_lo<KS>(pv.s.xlo, i);
  Acc<KS> asw[2], asp[2], asgr[2], srho;
  AccV3<KS> sv;
  struct Nb {
    float4 x, v;
    float rho, p;
    int ph;
  };
  auto load = [&](int j) { return Nb{pv.s.x[j], pv.s.v[j], pv.s.rho[j], pv.t.p[j], pv.s.phase[j]}; };
  for_each_pair4(L, g, i, xi, load, [&](int j, const Nb d) {
    const int phj = d.ph;
    if (!is_fluid(static_cast<uint8_t>(phj))) return;
    const V3 rwf = pos_diff<KS>(xi, li, ld3(d.x), pv.s.xlo, j);
    const float r2 = norm2(rwf);
    if (r2 >= P.support2) return;
    const float w = kW(P.kernel, sqrtf(r2));
    const float rhoj = d.rho;
    const int k = pidx(static_cast<uint8_t>(phj));
    for (int q = 0; q < 2; ++q) {  // constant indices: the sums stay in registers
      if (q != k) continue;
      asw[q] += w;
      asp[q] += d.p * w;
      asgr[q] += dot(grav, rwf) * rhoj * w;
    }
    srho += rhoj * w;
    sv += ld3(d.v) * w;
  });
  const float sw[2] = {float(asw[0]), float(asw[1])};
  const float sp[2] = {float(asp[0]), float(asp[1])}, sgr[2] = {float(asgr[0]), float(asgr[1])};
  float pw[2];
  for (int k = 0; k < 2; ++k) {
    pw[k] = sw[k] > 0.0f ? (sp[k] + sgr[k]) / sw[k] : P.p_bg;
    if (P.clamp_neg && pw[k] < 0.0f) pw[k] = 0.0f;
  }
  if (!(sw[0] > 0.0f) && sw[1] > 0.0f) pw[0] = pw[1];
  if (!(sw[1] > 0.0f) && sw[0] > 0.0f) pw[1] = pw[0];
  pv.t.p[i] = pw[0];
  pv.t.p_wv[i] = pw[1];
  pv.t.alpha[i] = (sw[0] + sw[1]) > 0.0f ? sw[0] / (sw[0] + sw[1]) : 0.0f;
  const float swt = sw[0] + sw[1];
  float rho_w;
  if (swt > 0.0f) {
    rho_w = float(srho) / swt;
    pv.t.vw[i] = st3(V3(sv) * (-1.0f / swt));
  } else {
    rho_w = P.rho0[0];
    pv.t.vw[i] = st3(V3{0, 0, 0});
  }
  pv.s.rho[i] = rho_w;
  // Liquid targets' transport-velocity wall density (SPH_kernels.cu:56-104)
  // depends on this wall only: evaluated once here, not once per pair.
  float rho_tvf = rho_w;
  if (P.tvf) {
    const float ratio = (pw[0] - P.p_bg) / P.tait_B + 1.0f;
    rho_tvf = P.rho0[0] * powf_cr(ratio > 0.5f ? ratio : 0.5f, 1.0f / P.tait_gamma);
  }
  const float4 q = make_float4(pw[0], pw[1], rho_tvf, pv.s.T[i]);
  pv.t.vol[i] = rho_tvf;
  float4 ghost = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (P.no_slip && swt > 0.0f) ghost = st3(V3(sv) * (-1.0f / swt));
  pv.t.rec[i] = PairRec{make_float4(xi.x, xi.y, xi.z, __int_as_float(kWall)), q, ghost, st3(V3{0, 0, 0})};
  pv.t.a[i] = st3(V3{0, 0, 0});
}

// ------------------------------------------------------- interface fields
// What one neighbour contributes to the interface pass.  x.w holds the
// phase in bits 0-7 and the flags in bits 8-15.  Fluid: r.x = m / rho.
// Wall: r = {nrm, alpha} (alpha only when walls carry a colour).  v: the
// fluid velocity or the wall's ghost velocity (SPS only).
struct IfaceNbr {
  float4 x, r, v;
};

template <bool SPS>
__device__ inline IfaceNbr load_iface_nbr(const PV& pv, const SimParams& P, int j) {
  IfaceNbr d;
  const float4 x = pv.s.x[j];
  const int ph = pv.s.phase[j];
  const int fl = pv.s.flags[j];
  d.x = make_float4(x.x, x.y, x.z, __int_as_float(ph | (fl << 8)));
  d.v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (ph == kWall) {
    const float4 nw = pv.s.nrm[j];
    // (fluid alpha is being written by this pass: walls' only)
    d.r = make_float4(nw.x, nw.y, nw.z, P.wall_colour ? pv.t.alpha[j] : 0.0f);
    if (SPS && P.no_slip) d.v = pv.t.vw[j];
  } else {
    d.r = make_float4(pv.t.vol[j], 0.0f, 0.0f, 0.0f);  // m / rho (density pass)
    if (SPS) d.v = pv.s.v[j];
  }
  return d;
}

// The interface fields of fluid particle i from its sums.
__device__ inline void interface_finish(const PV& pv, const SimParams& P, int i, uint8_t ph, int csf_mode, V3 gradc,
                                        V3 wall_n, V3 akn, V3 gradphi, float s_all, float s_other, float ww,
                                        float hw) {
  pv.t.alpha[i] = s_all > 0.0f ? s_other / s_all : 0.0f;
  pv.t.wall_w[i] = ww;
  pv.t.heat_w[i] = hw;
  if (P.st_model == 2) {
    pv.s.nrm[i] = st3(ph == kLiquid ? akn * (-P.kernel.h) : V3{0, 0, 0});
  } else {
    const float gmag = norm(gradc);
    V3 vwi{0, 0, 0};
    if (P.wetting != 0 && ww > 0.0f && gmag > P.normal_eps && norm2(wall_n) > 0.0f) {
      const V3 nw = normalized(wall_n);
      const V3 nh = gradc / gmag;
      const V3 tan_in = nh - nw * dot(nh, nw);
      const float tm = norm(tan_in);
      if (tm > 1e-6f) {
        const float cos_d = -dot(nh, nw);
        const float delta_w = 2.0f * norm(gradphi);
        const float coeff = 2.0f * P.sigma / (P.rho0[0] + P.rho0[1]);
        vwi = tan_in * (-(P.cos_theta - cos_d) * coeff * gmag * delta_w / tm);
      }
    }
    pv.t.vw[i] = st3(vwi);
    if (P.wetting != 1 && ww > 0.0f && gmag > P.normal_eps) {
      const V3 nw = normalized(wall_n);
      const V3 nh = gradc / gmag;
      V3 t = nh - nw * dot(nh, nw);
      const float tmag = norm(t);
      if (norm2(nw) > 0.0f && tmag > 1e-6f) {
        t = t / tmag;
        const V3 target = nw * (-P.cos_theta) + t * P.sin_theta;
        const float beta = clampv(ww / P.wall_adh_w, 0.0f, 1.0f);
        const V3 blended = normalized(nh * (1.0f - beta) + target * beta);
        gradc = blended * gmag;
      }
    }
    pv.s.nrm[i] = st3(gradc);
    if (csf_mode && !P.csf_smooth) {
      const float gm = norm(gradc);
      pv.t.ns[i] = st3(!(gm > P.normal_eps) ? V3{0, 0, 0} : gradc / gm);
    }
  }
}

// compute_interface_fields (surface_tension.cu:5-85) + SPS (navier_stokes.cu:
// 71-119) + normals without smoothing (surface_tension.cu:87-118) for particle
// i; returns its heat weight (0 unless fluid).  visit(f): f(j, IfaceNbr) over
// the neighbours in the reference order.
template <bool SPS, bool KS, class Visit>
__device__ inline float interface_particle(const PV& pv, const SimParams& P, int i, int csf_mode, Visit&& visit) {
  const uint8_t ph = pv.s.phase[i];
  if (!is_fluid(ph)) {
    if (SPS) pv.t.nu_t[i] = 0.0f;
    return 0.0f;
  }
  const V3 xi = ld3(pv.s.x[i]);
  const V3 li = pos_lo<KS>(pv.s.xlo, i);
  const float ci = ph == kLiquid ? 1.0f : 0.0f;
  AccV3<KS> agradc, awall_n, aakn, agradphi;
  Acc<KS> as_all, as_other, aww, ahw;
  const V3 vi = ld3(pv.s.v[i]);
  Acc<KS> Lm[3][3];
  visit([&](int j, const IfaceNbr d) {
    const V3 rij = pos_diff<KS>(xi, li, ld3(d.x), pv.s.xlo, j);
    const float r2 = norm2(rij);
    if (r2 >= P.support2) return;
    const float r = sqrtf(r2);
    const float w = kW(P.kernel, r);
    const int bits = __float_as_int(d.x.w);
    const int phj = bits & 0xff;
    const V3 gw = kgradW(P.kernel, rij, r);
    if (SPS && j != i && !(phj == kWall && !P.no_slip)) {
      const V3 vj = ld3(d.v);
      const float Vj = phj == kWall ? P.vol0 : d.r.x;
      const V3 dv = (vj - vi) * Vj;
      const float dvc[3] = {dv.x, dv.y, dv.z};
      const float gwc[3] = {gw.x, gw.y, gw.z};
      for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) Lm[a][b] += dvc[a] * gwc[b];
    }
    if (phj == kWall) {
      const float vw = P.vol0 * w;
      aww += vw;
      if ((bits >> 8) & kHeated) ahw += vw;
      awall_n += ld3(d.r) * vw;
      agradphi += gw * P.vol0;
      if (P.wall_colour) agradc += gw * (P.vol0 * (d.r.w - ci));
      return;
    }
    const float Vj = d.r.x;
    as_all += Vj * w;
    if (phj != ph) as_other += Vj * w;
    if (j == i) return;
    const float cj = phj == kLiquid ? 1.0f : 0.0f;
    agradc += gw * (Vj * (cj - ci));
    if (phj == kLiquid) aakn += gw * Vj;
  });
  const float s_all = as_all, s_other = as_other, ww = aww, hw = ahw;
  if (SPS) {
    float ss = 0.0f;
    for (int a = 0; a < 3; ++a)
      for (int b = 0; b < 3; ++b) {
        const float sab = 0.5f * (float(Lm[a][b]) + float(Lm[b][a]));
        ss += sab * sab;
      }
    const float smag = sqrtf(2.0f * ss);
    const float l = P.smag_cs * P.dx;
    pv.t.nu_t[i] = l * l * smag;
  }
  interface_finish(pv, P, i, ph, csf_mode, agradc, awall_n, aakn, agradphi, s_all, s_other, ww, hw);
  return hw;
}

// The interface pass for runs without SPS or Akinci, skipping what is
// provably zero.  A neighbour of the particle's own phase adds exact zeros
// (c_J - c_I = 0 to the colour gradient, nothing to alpha's numerator), so a
// particle with neither a wall nor the other phase in its 27 cells gets the
// outputs of an empty sum directly.  Without vapour at all, a wall within 2h
// of a liquid particle has colour alpha_w = 1 and so adds zeros too: only wall
// neighbours are summed.  Bitwise the full pass's results (adding a zero to a
// running sum that starts at +0 never changes it).  Resets the dt maxima.
// A row of 16 lanes per particle that has a wall or the other phase nearby, up
// to kInterfaceLanes particles (kInterfaceLanesKs in the precision form, whose
// compensated additions cost four times a plain one and are repeated by all 16
// lanes): 13 ordered sums.  A block takes one particle per row: spans of 64, and
// with them four particles in turn for some rows, took 78 us at 70 k.
// us with the row / with one thread per particle, two-phase spheres:
//   plain  6 k 16 / 78, 26 k 27 / 66, 60 k 46 / 72, 100 k 69 / 81, 140 k 86 / 87, 188 k 106 / 87
//   precise  6 k 40 / 130, 20 k 71 / 101, 26 k 100 / 101, 45 k 120 / 105, 100 k 224 / 120
constexpr int kInterfaceLanes = 140000, kInterfaceLanesKs = 25000;
template <bool KS, int G>
__global__ __launch_bounds__(kBlock) void k_interface_lanes(PV pv, GridDev g, SimParams P, NbrList L, DevState* st,
                                                            Count nc, int csf_mode) {
  constexpr int span = kBlock / G;
  const int n = nc.get();
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (int k = 0; k < 5; ++k) st->max_bits[k] = 0u;
  }
  const int base = xcd_span(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x)) * span;
  if (base >= n) return;  // uniform over the block
  auto select = [&](int i) {
    const uint8_t ph = pv.s.phase[i];
    if (!is_fluid(ph)) return false;
    if (cells_any(g, ld3(pv.s.x[i]), kCellWall | (ph == kLiquid ? kCellVapor : kCellLiquid))) return true;
    pv.t.alpha[i] = 0.0f;
    pv.t.wall_w[i] = 0.0f;
    pv.t.heat_w[i] = 0.0f;
    pv.t.vw[i] = st3(V3{0, 0, 0});
    pv.s.nrm[i] = st3(V3{0, 0, 0});
    if (csf_mode && !P.csf_smooth) pv.t.ns[i] = st3(V3{0, 0, 0});
    return false;
  };
  for_each_group<G>(base, span, n, select, [&](int i, int sub) {
    const uint8_t ph = pv.s.phase[i];
    const V3 xi = ld3(pv.s.x[i]);
    const V3 li = pos_lo<KS>(pv.s.xlo, i);
    const float ci = ph == kLiquid ? 1.0f : 0.0f;
    // colour gradient, wall normal, wall gradient (x, y, z each), alpha's
    // denominator and numerator, wall and heater weights
    Acc<KS> a[13];
    lane_sums<G>(L, g, i, xi, sub, a, [&](int j, float (&t)[13]) {
      // the gathers in flight together (a wall's normal and colour only for
      // walls: this pass writes the fluid ones)
      const int phj = pv.s.phase[j], flags = pv.s.flags[j];
      const float4 xj = pv.s.x[j];
      const float Vj = pv.t.vol[j];
      settle(phj, flags, xj.x, xj.y, xj.z, Vj);
      if (!P.has_vapor && phj != kWall) return;
      const V3 rij = pos_diff<KS>(xi, li, ld3(xj), pv.s.xlo, j);
      const float r2 = norm2(rij);
      if (r2 >= P.support2) return;
      const float r = sqrtf(r2);
      const float w = kW(P.kernel, r);
      const V3 gw = kgradW(P.kernel, rij, r);
      if (phj == kWall) {
        const float vw = P.vol0 * w;
        t[11] = vw;
        if (flags & kHeated) t[12] = vw;
        const V3 nw = ld3(pv.s.nrm[j]) * vw;
        t[3] = nw.x, t[4] = nw.y, t[5] = nw.z;
        const V3 gp = gw * P.vol0;
        t[6] = gp.x, t[7] = gp.y, t[8] = gp.z;
        if (P.wall_colour) {
          const V3 gc = gw * (P.vol0 * (pv.t.alpha[j] - ci));
          t[0] = gc.x, t[1] = gc.y, t[2] = gc.z;
        }
        return;
      }
      t[9] = Vj * w;
      if (phj != ph) t[10] = Vj * w;
      if (j == i) return;
      const float cj = phj == kLiquid ? 1.0f : 0.0f;
      const V3 gc = gw * (Vj * (cj - ci));
      t[0] = gc.x, t[1] = gc.y, t[2] = gc.z;
    });
    if (sub == 0)
      interface_finish(pv, P, i, ph, csf_mode, V3{float(a[0]), float(a[1]), float(a[2])},
                       V3{float(a[3]), float(a[4]), float(a[5])}, V3{0, 0, 0},
                       V3{float(a[6]), float(a[7]), float(a[8])}, float(a[9]), float(a[10]), float(a[11]),
                       float(a[12]));
  });
}

// The same with one thread per particle (many particles); also writes the heat
// partials.
template <bool KS>
__global__ __launch_bounds__(kBlock) void k_interface_sparse(PV pv, GridDev g, SimParams P, NbrList L, DevState* st,
                                                            Count nc, int csf_mode, double* heat_partials) {
  const int n = nc.get();
  const int i = gtid();
  if (i == 0) {
    for (int k = 0; k < 5; ++k) st->max_bits[k] = 0u;
  }
  double heat_contrib = 0.0;
  const uint8_t ph = i < n ? pv.s.phase[i] : kDead;
  if (is_fluid(ph)) {
    const V3 xi = ld3(pv.s.x[i]);
    if (cells_any(g, xi, kCellWall | (ph == kLiquid ? kCellVapor : kCellLiquid))) {
      if (P.has_vapor) {
        auto all = [&](auto&& f) {
          for_each_pair(L, g, i, xi, [&](int j) { f(j, load_iface_nbr<false>(pv, P, j)); });
        };
        heat_contrib = static_cast<double>(interface_particle<false, KS>(pv, P, i, csf_mode, all));
      } else {
        auto walls = [&](auto&& f) {
          for_each_pair(L, g, i, xi, [&](int j) {
            if (pv.s.phase[j] == kWall) f(j, load_iface_nbr<false>(pv, P, j));
          });
        };
        heat_contrib = static_cast<double>(interface_particle<false, KS>(pv, P, i, csf_mode, walls));
      }
    } else {
      pv.t.alpha[i] = 0.0f;
      pv.t.wall_w[i] = 0.0f;
      pv.t.heat_w[i] = 0.0f;
      pv.t.vw[i] = st3(V3{0, 0, 0});
      pv.s.nrm[i] = st3(V3{0, 0, 0});
      if (csf_mode && !P.csf_smooth) pv.t.ns[i] = st3(V3{0, 0, 0});
    }
  }
  if (heat_partials) block_sum_store(heat_contrib, heat_partials + blockIdx.x);
}

// Global-memory instance.  only_overflow = 0: every particle, resets the dt
// maxima for k_forces and writes FP64 block partials of sum_fluid heat_w
// (sph_solver.cu:101-104) when heat_partials != nullptr.  only_overflow = 1:
// just the particles whose list overflowed (the cell-tile instance does the
// rest).
template <bool SPS, bool KS>
__global__ __launch_bounds__(kBlock) void k_interface(PV pv, GridDev g, SimParams P, NbrList L, DevState* st, Count nc,
                                                     int csf_mode, double* heat_partials, int only_overflow) {
  const int n = nc.get();
  const int i = gtid();
  if (i == 0 && !only_overflow) {
    for (int k = 0; k < 5; ++k) st->max_bits[k] = 0u;
  }
  double heat_contrib = 0.0;
  if (i < n && (!only_overflow || (L.valid && L.count[i] < 0))) {
    const V3 xi = ld3(pv.s.x[i]);
    auto gathered = [&](auto&& f) {
      for_each_pair(L, g, i, xi, [&](int j) { f(j, load_iface_nbr<SPS>(pv, P, j)); });
    };
    heat_contrib = static_cast<double>(interface_particle<SPS, KS>(pv, P, i, csf_mode, gathered));
  }
  if (heat_partials) block_sum_store(heat_contrib, heat_partials + blockIdx.x);
}

// surface_tension.cu:87-118 with neighbour smoothing on.
template <bool KS>
__global__ __launch_bounds__(kBlock) void k_smooth_normals(PV pv, GridDev g, SimParams P, NbrList L, Count nc) {
  const int n = nc.get();
  const int i = gtid();
  if (i >= n) return;
  if (!is_fluid(pv.s.phase[i])) return;
  const V3 gi = ld3(pv.s.nrm[i]);
  const float gmag = norm(gi);
  if (!(gmag > P.normal_eps)) {
    pv.t.ns[i] = st3(V3{0, 0, 0});
    return;
  }
  const V3 xi = ld3(pv.s.x[i]);
  const V3 li = pos_lo<KS>(pv.s.xlo, i);
  AccV3<KS> acc;
  for_each_pair(L, g, i, xi, [&](int j) {
    if (!is_fluid(pv.s.phase[j])) return;
    const V3 gj = ld3(pv.s.nrm[j]);
    const float gjm = norm(gj);
    if (!(gjm > P.normal_eps)) return;
    const float r2 = norm2(pos_diff<KS>(xi, li, ld3(pv.s.x[j]), pv.s.xlo, j));
    if (r2 >= P.support2) return;
    acc += gj * ((pv.s.m[j] / pv.s.rho[j]) * kW(P.kernel, sqrtf(r2)) / gjm);
  });
  pv.t.ns[i] = st3(normalized(V3(acc)));
}

// ------------------------------------------------------ LDS-staged cell tiles
// One workgroup per tile of 3 x 3 x 3 cells.  Every neighbour of the tile's
// particles lies in the 5 x 5 x 5 cells around it: up to 25 (z, y) rows, each
// one contiguous index range of the cell-sorted arrays.  The workgroup copies
// those rows' neighbour data into LDS once (coalesced), then each thread
// walks its particle's neighbour list reading LDS.  List entries ascend, so a
// forward-moving row cursor maps index j to its LDS slot.  A tile whose rows
// hold more than kTileCap particles gathers from global memory instead;
// overflowed lists (count < 0) are left to the overflow instance of k_interface.
// The tile shape (g.tx x g.ty x g.tz cells, 3 x 3 x 3 by default) is a launch
// parameter: any shape with (ty + 2)(tz + 2) <= kTileRows staged rows and
// ty tz <= kTileTargetRows target rows (tile_shape_ok) gives the same results.
constexpr int kTileThreads = 512;
constexpr int kTileCap = 2304;
constexpr int kTileRows = 25;
constexpr int kTileTargetRows = 9;

struct TileRows {
  int start[kTileRows];     // first sorted index of each staged row
  int base[kTileRows + 1];  // its first LDS slot (exclusive prefix of row lengths)
  int rend[kTileRows];      // start + length: first sorted index after the row
  int roff[kTileRows];      // base - start: slot = j + roff for j in the row
  int nrows;
  int tstart[kTileTargetRows];  // the tile's own rows (targets)
  int tbase[kTileTargetRows + 1];
  int ntrows;
};

// Number of cell tiles (workgroups) of the tiled passes over grid g.
inline long long tile_count(const GridDev& g) {
  if (!tile_shape_ok(g.tx, g.ty, g.tz)) throw std::logic_error("cell-tile shape out of range");
  return static_cast<long long>((g.nx + g.tx - 1) / g.tx) * ((g.ny + g.ty - 1) / g.ty) * ((g.nz + g.tz - 1) / g.tz);
}

// Row tables of tile `b`; called by the whole block, ends with a barrier.
__device__ inline void tile_rows(const GridDev& g, int b, TileRows& T) {
  const int tiles_x = (g.nx + g.tx - 1) / g.tx;
  const int tiles_y = (g.ny + g.ty - 1) / g.ty;
  const int cx0 = (b % tiles_x) * g.tx;
  const int cy0 = ((b / tiles_x) % tiles_y) * g.ty;
  const int cz0 = (b / (tiles_x * tiles_y)) * g.tz;
  const int cx1 = min(cx0 + g.tx, g.nx), cy1 = min(cy0 + g.ty, g.ny), cz1 = min(cz0 + g.tz, g.nz);
  const int sx0 = max(cx0 - 1, 0), sx1 = min(cx1, g.nx - 1);
  const int sy0 = max(cy0 - 1, 0), sy1 = min(cy1, g.ny - 1);
  const int sz0 = max(cz0 - 1, 0), sz1 = min(cz1, g.nz - 1);
  const int nyr = sy1 - sy0 + 1;
  const int nrows = (sz1 - sz0 + 1) * nyr;
  const int tyr = cy1 - cy0;
  const int ntrows = (cz1 - cz0) * tyr;
  const int t = threadIdx.x;
  // row lengths in parallel: threads [0, nrows) staged rows (nrows <= 25),
  // [32, 32 + ntrows) target rows (ntrows <= 9)
  int first = 0, len = 0;
  if (t < nrows) {
    const int row = ((sz0 + t / nyr) * g.ny + (sy0 + t % nyr)) * g.nx;
    first = g.off[row + sx0];
    len = g.off[row + sx1 + 1] - first;
    T.start[t] = first;
  } else if (t >= 32 && t < 32 + ntrows) {
    const int k = t - 32;
    const int row = ((cz0 + k / tyr) * g.ny + (cy0 + k % tyr)) * g.nx;
    first = g.off[row + cx0];
    len = g.off[row + cx1] - first;
    T.tstart[k] = first;
  }
  // prefix sums of the row lengths within wave 0 (staged rows) and its upper half (target rows)
  if (t < 64) {
    int v = len;
    for (int off = 1; off < 32; off <<= 1) {
      const int o = __shfl_up(v, off, 32);
      if ((t & 31) >= off) v += o;
    }
    if (t < nrows) {
      T.base[t + 1] = v;
      T.rend[t] = first + len;
      T.roff[t] = v - len - first;
    } else if (t >= 32 && t < 32 + ntrows) {
      T.tbase[t - 32 + 1] = v;
    }
    if (t == 0) {
      T.base[0] = T.tbase[0] = 0;
      T.nrows = nrows;
      T.ntrows = ntrows;
    }
  }
  __syncthreads();
}

// Maps a particle's ascending list entries to LDS slots: the row of the
// current entry is kept with its end and offset, and only an entry past the
// row's end moves it forward.
struct RowCursor {
  const TileRows& T;
  int r, rend, roff;
  __device__ explicit RowCursor(const TileRows& t) : T(t), r(0), rend(t.rend[0]), roff(t.roff[0]) {}
  __device__ inline int slot(int j) {
    while (j >= rend && r < T.nrows - 1) {
      ++r;
      rend = T.rend[r];
      roff = T.roff[r];
    }
    return j + roff;
  }
};

// Sorted index of LDS slot s of a tile (s < the tile's staged count).
__device__ inline int tile_slot_index(const TileRows& T, int s) {
  int lo = 0, hi = T.nrows - 1;  // last row with base <= s
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (T.base[mid] <= s) lo = mid;
    else hi = mid - 1;
  }
  return T.start[lo] + (s - T.base[lo]);
}
// Slots a thread stages: every load of all of them is issued before the
// first one is waited for (one memory round trip per staging pass).
constexpr int kStageSlots = (kTileCap + kTileThreads - 1) / kTileThreads;

// One round of a tile's targets (round * kTileThreads + threadIdx.x): the
// fluid particles with a complete list go, in target order, to
// work[0, returned count); `other(i)` is called for the rest with a complete
// list (non-fluid: their zero outputs).  Overflowed lists are skipped (their
// own instance handles them).  Block-wide: every thread calls it.
template <class Other>
__device__ inline int tile_round_fluid(const PV& pv, const NbrList& L, const TileRows& T, int ntarget, int round,
                                       int* work, int* wave_tot, Other&& other) {
  const int t = round * kTileThreads + static_cast<int>(threadIdx.x);
  int i = -1;
  bool keep = false;
  if (t < ntarget) {
    int k = 0;
    while (t >= T.tbase[k + 1]) ++k;
    i = T.tstart[k] + (t - T.tbase[k]);
    if (L.count[i] >= 0) {
      if (is_fluid(pv.s.phase[i])) keep = true;
      else other(i);
    }
  }
  const unsigned long long mask = __ballot(keep);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  if (lane == 0) wave_tot[wave] = __popcll(mask);
  __syncthreads();
  int base = 0, total = 0;
  for (int w = 0; w < kTileThreads / 64; ++w) {
    const int c = wave_tot[w];
    base += w < wave ? c : 0;
    total += c;
  }
  if (keep) work[base + __popcll(mask & lt)] = i;
  __syncthreads();
  return total;
}


// ---------------------------------------------- interface, LDS-staged tiles
// Staged per particle: x with phase and flags bits, and {m/rho} (fluid) or {nrm, alpha} (wall): 32 B, so
// two workgroups fit a CU (48 B and one workgroup with SPS).  Wall normals
// and colours are staged for walls only: the pass writes the fluid ones.
// Writes heat_w, not its sum (k_heat_partials sums it).
template <bool SPS, bool KS>
__global__ __launch_bounds__(kTileThreads) void k_interface_tiled(PV pv, GridDev g, SimParams P, NbrList L,
                                                                DevState* st, int csf_mode) {
  __shared__ TileRows T;
  __shared__ float4 s_x[kTileCap], s_r[kTileCap], s_v[SPS ? kTileCap : 1];
  __shared__ int s_work[kTileThreads], s_wave[kTileThreads / 64];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (int k = 0; k < 5; ++k) st->max_bits[k] = 0u;
  }
  tile_rows(g, blockIdx.x, T);
  const int ntarget = T.tbase[T.ntrows];
  if (ntarget == 0) return;  // uniform over the block
  const int M = T.base[T.nrows];
  const bool staged = M <= kTileCap;
  // the first round's fluid targets are packed before staging: a tile of
  // walls alone stages nothing
  auto none = [](auto&&) {};
  auto other = [&](int i) { interface_particle<SPS, KS>(pv, P, i, csf_mode, none); };
  const int nfl0 = tile_round_fluid(pv, L, T, ntarget, 0, s_work, s_wave, other);
  if (nfl0 == 0 && ntarget <= kTileThreads) return;  // uniform over the block
  if (staged) {
    // Named slots, not arrays (arrays of them are not kept in registers).
    // First pass: position, phase, flags; second: what the phase selects (a
    // wall's normal and colour, a fluid particle's volume).
    struct Slot {
      float4 x, r, v;
      int j, bits;
      float a;
    };
    auto load1 = [&](int u) {
      Slot q{};
      const int s = threadIdx.x + u * kTileThreads;
      if (s < M) {
        q.j = tile_slot_index(T, s);
        q.x = pv.s.x[q.j];
        q.bits = static_cast<int>(pv.s.phase[q.j]) | (static_cast<int>(pv.s.flags[q.j]) << 8);
      }
      return q;
    };
    auto load2 = [&](int u, Slot q) {
      const int s = threadIdx.x + u * kTileThreads;
      if (s < M) {
        const bool wall = (q.bits & 0xff) == kWall;
        // (fluid normals and colours are being written by this pass)
        if (wall) q.r = pv.s.nrm[q.j];
        if (!wall || P.wall_colour) q.a = (wall ? pv.t.alpha : pv.t.vol)[q.j];  // two global arrays: a pointer select is fine
        q.v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (SPS && (!wall || P.no_slip)) q.v = (wall ? pv.t.vw : pv.s.v)[q.j];
      }
      return q;
    };
    auto store = [&](int u, const Slot q) {
      const int s = threadIdx.x + u * kTileThreads;
      if (s < M) {
        const bool wall = (q.bits & 0xff) == kWall;
        s_x[s] = make_float4(q.x.x, q.x.y, q.x.z, __int_as_float(q.bits));
        s_r[s] = wall ? make_float4(q.r.x, q.r.y, q.r.z, q.a) : make_float4(q.a, 0.0f, 0.0f, 0.0f);
        if (SPS) s_v[s] = q.v;
      }
    };
    static_assert(kStageSlots == 5, "staging is written out for five slots per thread");
    Slot q0 = load1(0), q1 = load1(1), q2 = load1(2), q3 = load1(3), q4 = load1(4);
    q0 = load2(0, q0);
    q1 = load2(1, q1);
    q2 = load2(2, q2);
    q3 = load2(3, q3);
    q4 = load2(4, q4);
    store(0, q0);
    store(1, q1);
    store(2, q2);
    store(3, q3);
    store(4, q4);
  }
  __syncthreads();
  for (int round = 0; round * kTileThreads < ntarget; ++round) {
    const int nfl = round == 0 ? nfl0 : tile_round_fluid(pv, L, T, ntarget, round, s_work, s_wave, other);
    if (static_cast<int>(threadIdx.x) >= nfl) continue;
    const int i = s_work[threadIdx.x];
    const int cnt = L.count[i];
    if (staged) {
      auto from_lds = [&](auto&& f) {
        RowCursor rc(T);
        for_each_listed(L, i, cnt, [&](int j) {
          const int s = rc.slot(j);
          const float4 xs = s_x[s], rs = s_r[s];
          float4 vs = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
          if (SPS) vs = s_v[s];
          f(j, IfaceNbr{xs, rs, vs});
        });
      };
      interface_particle<SPS, KS>(pv, P, i, csf_mode, from_lds);
    } else {
      auto gathered = [&](auto&& f) {
        for_each_listed(L, i, cnt, [&](int j) { f(j, load_iface_nbr<SPS>(pv, P, j)); });
      };
      interface_particle<SPS, KS>(pv, P, i, csf_mode, gathered);
    }
  }
}

// FP64 block partials of sum_fluid heat_w (sph_solver.cu:101-104).
__global__ __launch_bounds__(kBlock) void k_heat_partials(PV pv, Count nc, double* partials) {
  const int n = nc.get();
  const int i = gtid();
  double v = 0.0;
  if (i < n && is_fluid(pv.s.phase[i])) v = static_cast<double>(pv.t.heat_w[i]);
  block_sum_store(v, partials + blockIdx.x);
}

// Publishes the maxima (spacing ratio starts from 1, sph_solver.cu:62-71).
__global__ void k_publish_maxima(DevState* st, int has_vapor, int sps) {
  st->v_max = __uint_as_float(st->max_bits[0]);
  st->a_max = __uint_as_float(st->max_bits[1]);
  st->Tv_max = has_vapor ? __uint_as_float(st->max_bits[2]) : 0.0f;
  st->nu_t_max = sps ? __uint_as_float(st->max_bits[3]) : 0.0f;
  const float sp = __uint_as_float(st->max_bits[4]);
  st->spacing_ratio = sp > 1.0f ? sp : 1.0f;
}

// sph_solver.cu:466-472: heat_inv_norm from the FP64 partials.
__global__ __launch_bounds__(1024) void k_heat_norm(DevState* st, const double* partials, int nb, int active) {
  __shared__ double s[1024];
  double acc = 0.0;
  for (int k = threadIdx.x; k < nb; k += 1024) acc += partials[k];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int off = 512; off > 0; off >>= 1) {
    if (static_cast<int>(threadIdx.x) < off) s[threadIdx.x] += s[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double S = s[0];
    st->heat_inv_norm = active ? (S > 0 ? static_cast<float>(1.0 / S) : 0.0f) : 0.0f;
  }
}

// probe_liquid_pressure (sph_solver.cu:197-216)
__global__ __launch_bounds__(kBlock) void k_probe(PV pv, GridDev g, SimParams P, const float* pts, float* out,
                                                 int np) {
  const int k = gtid();
  if (k >= np) return;
  const V3 x{pts[3 * k], pts[3 * k + 1], pts[3 * k + 2]};
  float num = 0.0f, den = 0.0f;
  for_each_nbr(g, x, [&](int j) {
    if (pv.s.phase[j] != kLiquid) return;
    const float r2 = norm2(x - ld3(pv.s.x[j]));
    if (r2 >= P.support2) return;
    const float w = (pv.s.m[j] / pv.s.rho[j]) * kW(P.kernel, sqrtf(r2));
    num += pv.t.p[j] * w;
    den += w;
  });
  out[k] = den > 0.0f ? num / den : __builtin_nanf("");
}

// SPH_kernels.cu:106-160 (delta+ shifting), pass 1 and pass 2.
template <bool KS>
__global__ __launch_bounds__(kBlock) void k_shift_compute(PV pv, GridDev g, SimParams P, NbrList L,
                                                         const DevState* st, Count nc) {
  const int n = nc.get();
  const int i = gtid();
  if (i >= n) return;
  pv.t.ns[i] = st3(V3{0, 0, 0});
  const uint8_t ph = pv.s.phase[i];
  if (!is_fluid(ph) || pv.t.sigma[i] < P.tvf_sigma_min) return;
  const float h = P.kernel.h;
  const float w_dx = kW(P.kernel, P.dx);
  const float mach = st->v_max / P.c0;
  const float coeff = P.shift_strength * mach * 4.0f * h * h;
  const float cap = 0.1f * P.dx;
  const V3 xi = ld3(pv.s.x[i]);
  const V3 li = pos_lo<KS>(pv.s.xlo, i);
  AccV3<KS> sum;
  for_each_pair(L, g, i, xi, [&](int j) {
    if (j == i) return;
    const uint8_t phj = pv.s.phase[j];
    if (phj == kDead) return;
    const V3 rij = pos_diff<KS>(xi, li, ld3(pv.s.x[j]), pv.s.xlo, j);
    const float r2 = norm2(rij);
    if (r2 >= P.support2) return;
    const float r = sqrtf(r2);
    const float Vj = phj == kWall ? 1.0f / pv.t.sigma[i] : 1.0f / pv.t.sigma[j];
    const float qq = kW(P.kernel, r) / w_dx;
    const float q2 = qq * qq;
    sum += kgradW(P.kernel, rij, r) * (Vj * (1.0f + 0.2f * q2 * q2));
  });
  V3 dr = V3(sum) * (-coeff);
  if (pv.t.alpha[i] > 0.0f) {
    const V3 gn = ld3(pv.s.nrm[i]);
    const float gm = norm(gn);
    if (gm > P.normal_eps) {
      const V3 nn = gn / gm;
      dr -= nn * dot(dr, nn);
    } else {
      dr = V3{0, 0, 0};
    }
  }
  const float len = norm(dr);
  if (len > cap) dr *= cap / len;
  pv.t.ns[i] = st3(dr);
}

__global__ __launch_bounds__(kBlock) void k_shift_apply(PV pv, Count nc) {
  const int n = nc.get();
  const int i = gtid();
  if (i >= n) return;
  if (!is_fluid(pv.s.phase[i])) return;
  if (pv.s.xlo) {  // precision form: the shift into the double-float position
    V3 x = ld3(pv.s.x[i]), lo = ld3(pv.s.xlo[i]);
    const V3 d = ld3(pv.t.ns[i]);
    df_add(x.x, lo.x, d.x);
    df_add(x.y, lo.y, d.y);
    df_add(x.z, lo.z, d.z);
    pv.s.x[i] = st3(x);
    pv.s.xlo[i] = st3(lo);
  } else {
    pv.s.x[i] = st3(ld3(pv.s.x[i]) + ld3(pv.t.ns[i]));
  }
}

}  // namespace

void launch_density(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, Count n, hipStream_t s) {
  if (n.ub <= 0) return;
  if (n.ub >= kDensWide) {
    if (P.compensated) k_density_wide<true><<<blocks_for(n.ub), kBlock, 0, s>>>(pv, g, P, L, n);
    else k_density_wide<false><<<blocks_for(n.ub), kBlock, 0, s>>>(pv, g, P, L, n);
    return;
  }
  const int nb = blocks_for(static_cast<long long>(n.ub) * kDensLanes);
  if (P.compensated) k_density<true><<<nb, kBlock, 0, s>>>(pv, g, P, L, n);
  else k_density<false><<<nb, kBlock, 0, s>>>(pv, g, P, L, n);
}
void launch_normalize_masses(const PV& pv, const GridDev& g, const SimParams& P, int n, hipStream_t s) {
  if (n <= 0) return;
  if (P.compensated) k_normalize_masses<true><<<blocks_for(n), kBlock, 0, s>>>(pv, g, P, n);
  else k_normalize_masses<false><<<blocks_for(n), kBlock, 0, s>>>(pv, g, P, n);
}
void launch_wall_bc(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, const DevState* st, Count n,
                    hipStream_t s) {
  if (n.ub <= 0) return;
  if (P.compensated) k_wall_bc<true><<<blocks_for(n.ub), kBlock, 0, s>>>(pv, g, P, L, st, n);
  else k_wall_bc<false><<<blocks_for(n.ub), kBlock, 0, s>>>(pv, g, P, L, st, n);
}
template <bool SPS, bool KS>
static void interface_variant(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, DevState* st,
                              Count n, int cm, double* heat_partials, bool tiled, hipStream_t s) {
  const int nb = blocks_for(n.ub > 0 ? n.ub : 1);
  if (!tiled) {
    k_interface<SPS, KS><<<nb, kBlock, 0, s>>>(pv, g, P, L, st, n, cm, heat_partials, 0);
    return;
  }
  const long long tiles = tile_count(g);
  if (tiles > 0x7fffffffLL) throw std::runtime_error("interface pass: too many cell tiles");
  k_interface_tiled<SPS, KS><<<static_cast<int>(tiles), kTileThreads, 0, s>>>(pv, g, P, L, st, cm);
  k_interface<SPS, KS><<<nb, kBlock, 0, s>>>(pv, g, P, L, st, n, cm, nullptr, 1);
  if (heat_partials) k_heat_partials<<<nb, kBlock, 0, s>>>(pv, n, heat_partials);
}
int launch_interface(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, DevState* st, Count n,
                     bool csf_mode, double* heat_partials, bool tiled, hipStream_t s) {
  const int nb = blocks_for(n.ub > 0 ? n.ub : 1);
  const int cm = csf_mode ? 1 : 0;
  if (!interface_has_tiles(P) && L.valid && g.flags) {
    if (n.ub < (P.compensated ? kInterfaceLanesKs : kInterfaceLanes)) {
      const int sb = blocks_for(16ll * std::max(n.ub, 1));
      if (P.compensated) k_interface_lanes<true, 16><<<sb, kBlock, 0, s>>>(pv, g, P, L, st, n, cm);
      else k_interface_lanes<false, 16><<<sb, kBlock, 0, s>>>(pv, g, P, L, st, n, cm);
      if (heat_partials) k_heat_partials<<<nb, kBlock, 0, s>>>(pv, n, heat_partials);
    } else {
      if (P.compensated) k_interface_sparse<true><<<nb, kBlock, 0, s>>>(pv, g, P, L, st, n, cm, heat_partials);
      else k_interface_sparse<false><<<nb, kBlock, 0, s>>>(pv, g, P, L, st, n, cm, heat_partials);
    }
    return nb;
  }
  tiled = tiled && L.valid;
  if (P.compensated) {
    if (P.sps) interface_variant<true, true>(pv, g, P, L, st, n, cm, heat_partials, tiled, s);
    else interface_variant<false, true>(pv, g, P, L, st, n, cm, heat_partials, tiled, s);
  } else {
    if (P.sps) interface_variant<true, false>(pv, g, P, L, st, n, cm, heat_partials, tiled, s);
    else interface_variant<false, false>(pv, g, P, L, st, n, cm, heat_partials, tiled, s);
  }
  return nb;
}
void launch_smooth_normals(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, Count n,
                           hipStream_t s) {
  if (n.ub <= 0) return;
  if (P.compensated) k_smooth_normals<true><<<blocks_for(n.ub), kBlock, 0, s>>>(pv, g, P, L, n);
  else k_smooth_normals<false><<<blocks_for(n.ub), kBlock, 0, s>>>(pv, g, P, L, n);
}
void launch_heat_norm(DevState* st, const double* partials, int nb, bool active, hipStream_t s) {
  k_heat_norm<<<1, 1024, 0, s>>>(st, partials, nb, active ? 1 : 0);
}

// Lanes per particle of the forces pass: four while the chip is not full
// (shorter chains), two beyond (each lane of a group repeats the ordered
// additions, four times as dear in the precision form).  us with four / two,
// tanks and columns in motion:
//   CSF  45 k 56 / 73, 60 k 66 / 80, 75 k 81 / 84, 90 k 87 / 83, 188 k 149 / 145, 600 k 403 / 356
//   CSF, precise  26 k 68 / 88, 50 k 87 / 91, 60 k 115 / 100, 120 k 180 / 151, 600 k 682 / 513
//   no tension  76 k 45 / 59, 123 k 73 / 70, 150 k 74 / 78, 233 k 103 / 106, 297 k 130 / 124
//   no tension, SPS  76 k 55 / 71, 90 k 73 / 73, 123 k 88 / 83, 151 k 102 / 91, 233 k 139 / 143, 297 k 176 / 158
//   Akinci  90 k 133 / 156, 136 k 183 / 190, 256 k 302 / 312, 345 k 391 / 379
// `other` takes the other count.
int forces_lanes(const SimParams& P, bool csf_mode, int n, bool other) {
  const int below = P.compensated ? 50000 : csf_mode || P.sps ? 80000 : 250000;
  return (n < below) != other ? 4 : 2;
}

void launch_forces(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, DevState* st, Count n,
                   bool csf_mode, bool akinci, bool continuity, bool thermal, bool other_lanes, hipStream_t s) {
  const int lanes = forces_lanes(P, csf_mode, n.ub, other_lanes);
  if (akinci) launch_forces_akinci(pv, g, P, L, st, n, continuity, thermal, lanes, s);
  else if (csf_mode) launch_forces_csf(pv, g, P, L, st, n, continuity, thermal, lanes, s);
  else launch_forces_none(pv, g, P, L, st, n, continuity, thermal, lanes, s);
  k_publish_maxima<<<1, 1, 0, s>>>(st, P.has_vapor, P.sps);
}
void launch_probe(const PV& pv, const GridDev& g, const SimParams& P, const float* pts, float* out, int np,
                  hipStream_t s) {
  if (np > 0) k_probe<<<blocks_for(np), kBlock, 0, s>>>(pv, g, P, pts, out, np);
}
void launch_shifting(const PV& pv, const GridDev& g, const SimParams& P, const NbrList& L, const DevState* st, Count n,
                     hipStream_t s) {
  if (n.ub <= 0) return;
  if (P.compensated) k_shift_compute<true><<<blocks_for(n.ub), kBlock, 0, s>>>(pv, g, P, L, st, n);
  else k_shift_compute<false><<<blocks_for(n.ub), kBlock, 0, s>>>(pv, g, P, L, st, n);
  k_shift_apply<<<blocks_for(n.ub), kBlock, 0, s>>>(pv, n);
}

}  // namespace cryo
