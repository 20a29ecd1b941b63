// SPME charge spread and force gather for gfx950, deterministic
// owner-computes mesh accumulation (no global atomics on the mesh).
//
// Reference behaviour: kernels/spme_spread_gather.cuh (Cox-de Boor weights
// :36-86, per-particle setup :90-126, spread :162-221, gather :227-334) and
// kernels/spme_recip.cu:208-253.  The reference spreads with p threads per
// atom and one global i64 atomic per mesh contribution.  Here:
//
//  * every step the atoms are binned by the mesh brick (b0 x b1 x b2 points)
//    that holds their primary point g = floor(u);
//  * one workgroup owns one brick: it walks the atoms of its own bin and of
//    the +1 neighbour bins along each axis (the only atoms whose p^3 support
//    reaches the brick, since b >= p), accumulates their contributions for
//    the points it owns in LDS as i64 fixed point (2^32, round to nearest,
//    as spme_spread_gather.cuh:211-212), and writes the brick once as f32.
//    Integer LDS sums make the result independent of atom order;
//  * the gather stages the brick's potential plus its (p-1) halo in LDS and
//    evaluates each atom of the brick's own bin in one thread.
#include "hmd_device.h"

template <int P>
__device__ inline void hmd_bspline(float x, float w[P]) {
  // M_P(x - 0 .. x - (P-1)) by Cox-de Boor from the M_1 indicators; returns
  // w[d] = M_P(d + t) for x = t, d = 0..P-1, evaluated as in
  // spme_spread_gather.cuh:36-54 (one recursion per support point).
#pragma unroll
  for (int d = 0; d < P; ++d) {
    float xd = x + (float)d;
    float v[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
      float xi = xd - (float)i;
      v[i] = (xi >= 0.0f && xi < 1.0f) ? 1.0f : 0.0f;
    }
#pragma unroll
    for (int order = 2; order <= P; ++order) {
      float inv = 1.0f / (float)(order - 1);
#pragma unroll
      for (int i = 0; i < P - order + 1; ++i) {
        float xi = xd - (float)i;
        v[i] = xi * inv * v[i] + ((float)order - xi) * inv * v[i + 1];
      }
    }
    w[d] = v[0];
  }
}

template <int P>
__device__ inline void hmd_bspline_deriv(float x, float w[P], float dw[P]) {
  // M_P(d + t) and M_P'(d + t) = M_{P-1}(d + t) - M_{P-1}(d + t - 1)
  // (spme_spread_gather.cuh:58-86).
#pragma unroll
  for (int d = 0; d < P; ++d) {
    float xd = x + (float)d;
    float v[P + 1];
#pragma unroll
    for (int i = 0; i < P + 1; ++i) {
      float xi = xd - (float)i;
      v[i] = (xi >= 0.0f && xi < 1.0f) ? 1.0f : 0.0f;
    }
#pragma unroll
    for (int order = 2; order < P; ++order) {
      float inv = 1.0f / (float)(order - 1);
#pragma unroll
      for (int i = 0; i < P - order + 1; ++i) {
        float xi = xd - (float)i;
        v[i] = xi * inv * v[i] + ((float)order - xi) * inv * v[i + 1];
      }
    }
    dw[d] = v[0] - v[1];
    float inv = 1.0f / (float)(P - 1);
    w[d] = xd * inv * v[0] + ((float)P - xd) * inv * v[1];
  }
}

// Order 4 in closed form (the cubic cardinal B-spline on its four unit
// intervals; the same function as the recursion, fewer operations):
// w[d] = M_4(d + t), dw[d] = M_4'(d + t).
template <>
__device__ inline void hmd_bspline<4>(float t, float w[4]) {
  const float t2 = t * t, t3 = t2 * t, u = 1.0f - t;
  const float s6 = 1.0f / 6.0f;
  w[0] = t3 * s6;
  w[1] = (1.0f + 3.0f * t + 3.0f * t2 - 3.0f * t3) * s6;
  w[2] = (4.0f - 6.0f * t2 + 3.0f * t3) * s6;
  w[3] = u * u * u * s6;
}

template <>
__device__ inline void hmd_bspline_deriv<4>(float t, float w[4], float dw[4]) {
  hmd_bspline<4>(t, w);
  const float t2 = t * t, u = 1.0f - t;
  dw[0] = 0.5f * t2;
  dw[1] = 0.5f * (1.0f + 2.0f * t - 3.0f * t2);
  dw[2] = 0.5f * (3.0f * t2 - 4.0f * t);
  dw[3] = -0.5f * u * u;
}

// u = (s + 1/2) n, primary point g = floor(u) mod n, t = u - floor(u)
// (spme_spread_gather.cuh:90-126).
__device__ inline void hmd_spme_setup(float4 a, const HmdLattice& L,
                                      uint32_t n0, uint32_t n1, uint32_t n2,
                                      float t[3], int g[3]) {
  float x = a.x, y = a.y, z = a.z;
  int ia, ib, ic;
  hmd_wrap(x, y, z, ia, ib, ic, L);
  float s[3];
  hmd_cart_to_frac(x, y, z, L, s[0], s[1], s[2]);
  const uint32_t nn[3] = {n0, n1, n2};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    float u = (s[d] + 0.5f) * (float)nn[d];
    float f = floorf(u);
    t[d] = u - f;
    int gi = (int)f % (int)nn[d];
    if (gi < 0) gi += (int)nn[d];
    g[d] = gi;
  }
}

// Bin each atom by the brick holding its primary point.  Atoms are visited
// in the neighbour list's Hilbert order, so a wave's 64 atoms fall into a few
// bins: one atomic per (wave, bin) instead of one per atom.  The primary
// point is computed from the same f32 position the spread and the gather
// read (posq, not the list's image-shifted copy): an atom within a rounding
// of a box face can wrap to the other face from a shifted copy, and the
// gather would then look for its stencil outside the brick it is binned in.
__device__ inline uint32_t hmd_spme_bin_of(const SpmeBinParams& p, float4 pq) {
  float t[3];
  int g[3];
  hmd_spme_setup(pq, p.L, p.n0, p.n1, p.n2, t, g);
  return ((uint32_t)g[0] / p.b0 * p.nb1 + (uint32_t)g[1] / p.b1) * p.nb2 +
         (uint32_t)g[2] / p.b2;
}

__device__ __forceinline__ void hmd_spme_bin_body(const SpmeBinParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t s = hmd_bx * blockDim.x + threadIdx.x;
  const bool valid = s < p.n;
  uint32_t bin = HMD_SENTINEL;
  if (valid) {
    bin = hmd_spme_bin_of(p, reinterpret_cast<const float4*>(p.posq)[p.sorted_id[s]]);
    p.atom_bin[s] = bin;
  }
  uint64_t pending = __ballot(valid);
  while (pending) {
    const uint32_t leader = (uint32_t)__builtin_ctzll(pending);
    const uint32_t b = hmd_readlane(bin, leader);
    const uint64_t same = __ballot(valid && bin == b);
    if (hmd_lane() == leader) atomicAdd(&p.bin_count[b], (uint32_t)__builtin_popcountll(same));
    pending &= ~same;
  }
}
HMD_KERNEL(hmd_spme_bin, SpmeBinParams, 256)

// Scatter canonical atom ids into their bins.  The count array is driven
// back to zero (one atomicSub per (wave, bin) claims a block of positions).
__device__ __forceinline__ void hmd_spme_bin_scatter_body(const SpmeBinParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t s = hmd_bx * blockDim.x + threadIdx.x;
  const bool valid = s < p.n;
  const uint32_t lane = hmd_lane();
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const uint32_t bin = valid ? p.atom_bin[s] : HMD_SENTINEL;
  uint64_t pending = __ballot(valid);
  while (pending) {
    const uint32_t leader = (uint32_t)__builtin_ctzll(pending);
    const uint32_t b = hmd_readlane(bin, leader);
    const uint64_t same = __ballot(valid && bin == b);
    const uint32_t cnt = (uint32_t)__builtin_popcountll(same);
    uint32_t old = 0;
    if (lane == leader) old = atomicSub(&p.bin_count[b], cnt);
    old = hmd_readlane(old, leader);
    if (valid && bin == b) {
      const uint32_t rank = (uint32_t)__builtin_popcountll(same & lt_mask);
      p.bin_atoms[p.bin_start[b] + old - cnt + rank] = p.sorted_id[s];
    }
    pending &= ~same;
  }
}
HMD_KERNEL(hmd_spme_bin_scatter, SpmeBinParams, 256)

// The three launches of the binning (bin, scan, scatter) in one workgroup,
// for systems of at most HMD_SPME_BIN_SMALL atoms and 4,096 bins: an atom's
// rank in its bin comes from the LDS count, so one pass over the atoms is
// enough.  The launches were 4.5 + 4.7 + 6.5 us at 648 atoms, each waiting
// for the one before.
__device__ __forceinline__ void hmd_spme_bin_small_body(const SpmeBinParams& p,
                                                        const uint32_t hmd_bx,
                                                        const uint32_t hmd_gx) {
  __shared__ uint32_t s_bins[4096];
  __shared__ uint32_t s_wave[16];
  constexpr uint32_t U = HMD_SPME_BIN_SMALL / 1024u;
  const uint32_t t = threadIdx.x, lane = hmd_lane(), wave = t / HMD_WAVE;
  const uint32_t n_bins = p.nb0 * p.nb1 * p.nb2;
  reinterpret_cast<uint4*>(s_bins)[t] = make_uint4(0u, 0u, 0u, 0u);
  uint32_t id[U], bin[U], rank[U];
#pragma unroll
  for (uint32_t u = 0; u < U; ++u)
    id[u] = p.sorted_id[min(t + 1024u * u, p.n - 1u)];
  float4 pq[U];
#pragma unroll
  for (uint32_t u = 0; u < U; ++u) pq[u] = reinterpret_cast<const float4*>(p.posq)[id[u]];
  __syncthreads();
#pragma unroll
  for (uint32_t u = 0; u < U; ++u) {
    if (t + 1024u * u < p.n) {
      bin[u] = hmd_spme_bin_of(p, pq[u]);
      rank[u] = atomicAdd(&s_bins[bin[u]], 1u);
    }
  }
  __syncthreads();
  // exclusive scan, four bins a thread
  const uint4 v = reinterpret_cast<const uint4*>(s_bins)[t];
  const uint32_t sum = v.x + v.y + v.z + v.w;
  uint32_t incl = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t w = (uint32_t)__shfl_up((int)incl, (unsigned)o, HMD_WAVE);
    if (lane >= (uint32_t)o) incl += w;
  }
  if (lane == HMD_WAVE - 1) s_wave[wave] = incl;
  __syncthreads();
  uint32_t e = incl - sum;
  for (uint32_t w = 0; w < wave; ++w) e += s_wave[w];
  const uint32_t start[4] = {e, e + v.x, e + v.x + v.y, e + v.x + v.y + v.z};
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    s_bins[4u * t + k] = start[k];
    if (4u * t + k < n_bins) p.bin_start[4u * t + k] = start[k];
  }
  if (t == 0) p.bin_start[n_bins] = p.n;
  __syncthreads();
#pragma unroll
  for (uint32_t u = 0; u < U; ++u)
    if (t + 1024u * u < p.n) p.bin_atoms[s_bins[bin[u]] + rank[u]] = id[u];
}
HMD_KERNEL(hmd_spme_bin_small, SpmeBinParams, 1024)

// A contribution v (in units of 2^-24 e, |v| < 2^31) as the i64 count of
// 2^-32 e rounded to nearest, from two i32 roundings: r1 = rint(v), the
// remainder v - r1 (exact in f32, |.| <= 1/2) scaled by 2^8 and rounded,
// and r1 * 2^8 + r2 -- the same value as rounding v * 2^8 directly, without
// the long f32 -> i64 conversion sequence.
__device__ inline long long hmd_fixed32_of24(float v) {
  const float f1 = rintf(v);
  const int r1 = (int)f1;
  const int r2 = (int)rintf((v - f1) * 256.0f);
  return ((long long)r1 << 8) + (long long)r2;
}

// Queue entries of the spread: weights of 2 x 256 atoms at order 4 (27 KB
// beside the brick), of one round of candidates at the higher orders.
#define HMD_SPREAD_QUEUE(P) ((P) == 4 ? 512u : 256u)

// Spread of one brick per workgroup.
//
// The atoms of the eight bins are one candidate list (their ranges joined by a
// prefix), filtered a workgroup's width at a time: a candidate whose support
// reaches the brick (a third to a quarter of them) puts its weights and mesh
// position into an LDS queue.  The queue is then worked off P lanes an atom,
// lane d taking the support plane d of the fast axis, so that P lanes add to P
// consecutive mesh points, every lane has the same P^2 adds to do, and lanes
// of atoms that miss the brick do not idle through the adds of the others.
// The contributions are the same numbers in whatever order, and integer sums:
// the mesh does not depend on the split.
//
// Bound by the latency of the chain bins -> atoms -> positions -> LDS adds in
// small systems and by the LDS adds in large ones.  One thread an atom
// over the eight bins in turn, all P^3 adds its own, took 29.1 us at 648
// atoms on 24^3 (now 6.0), 31 us at 24,576 on 64^3 (11.6), 47 us at 196,608
// on 128^3 (42) and 111 us at 4,503 on 40^3 with order 6 (26).
template <int P>
__device__ inline void hmd_spread_body(const SpmeSpreadParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  constexpr uint32_t Q = HMD_SPREAD_QUEUE(P);
  extern __shared__ long long s_acc[];
  __shared__ float s_w[3][P][Q];          // weights; axis 0 times the charge
  __shared__ uint16_t s_at[3][Q];         // primary point relative to the brick
  __shared__ uint32_t s_n;
  const uint32_t bsz = p.b0 * p.b1 * p.b2;
  const uint32_t B = hmd_bx;
  const uint32_t B2 = B % p.nb2, B1 = (B / p.nb2) % p.nb1, B0 = B / (p.nb2 * p.nb1);
  const int o0 = (int)(B0 * p.b0), o1 = (int)(B1 * p.b1), o2 = (int)(B2 * p.b2);
  const uint32_t lane = hmd_lane();
  // ranges of the eight bins (every thread: wave-uniform loads)
  uint32_t beg[8], cum[9];
  cum[0] = 0;
#pragma unroll
  for (uint32_t nb = 0; nb < 8; ++nb) {
    // With a single brick along an axis the +1 neighbour is the brick
    // itself: visit it once.
    const bool skip = (p.nb0 == 1 && (nb & 4u)) || (p.nb1 == 1 && (nb & 2u)) ||
                      (p.nb2 == 1 && (nb & 1u));
    const uint32_t c0 = (B0 + ((nb >> 2) & 1u)) % p.nb0;
    const uint32_t c1 = (B1 + ((nb >> 1) & 1u)) % p.nb1;
    const uint32_t c2 = (B2 + (nb & 1u)) % p.nb2;
    const uint32_t bin = (c0 * p.nb1 + c1) * p.nb2 + c2;
    beg[nb] = p.bin_start[bin];
    cum[nb + 1] = cum[nb] + (skip ? 0u : p.bin_start[bin + 1] - beg[nb]);
  }
  const uint32_t total = cum[8];
  for (uint32_t k = threadIdx.x; k < bsz; k += blockDim.x) s_acc[k] = 0;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();

  for (uint32_t k0 = 0; k0 < total; k0 += blockDim.x) {
    const uint32_t k = k0 + threadIdx.x;
    bool in = false;
    float wa[P], wb[P], wc[P];
    uint32_t at[3];
    if (k < total) {
      uint32_t at_k = 0;
#pragma unroll
      for (uint32_t nb = 0; nb < 8; ++nb)
        if (k >= cum[nb] && k < cum[nb + 1]) at_k = beg[nb] + (k - cum[nb]);
      const uint32_t a = p.bin_atoms[at_k];
      const float4 pq = reinterpret_cast<const float4*>(p.posq)[a];
      float t[3];
      int g[3];
      hmd_spme_setup(pq, p.L, p.n0, p.n1, p.n2, t, g);
      // Does any of the P support planes along each axis fall in this brick?
      const int oo[3] = {o0, o1, o2};
      const uint32_t nn[3] = {p.n0, p.n1, p.n2}, bb[3] = {p.b0, p.b1, p.b2};
      in = pq.w != 0.0f;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const int u = g[d] - oo[d];
        at[d] = (uint32_t)(u + (u < 0 ? (int)nn[d] : 0));
        // planes at[d], at[d] - 1, ..., at[d] - (P - 1), wrapped: the first
        // inside the brick, or one of the others after it (or past the wrap)
        in = in && (at[d] < bb[d] + (uint32_t)(P - 1));
      }
      if (in) {
        hmd_bspline<P>(t[0], wa);
        hmd_bspline<P>(t[1], wb);
        hmd_bspline<P>(t[2], wc);
        const float q24 = pq.w * 16777216.0f;   // charge in 2^-24 units
#pragma unroll
        for (int d = 0; d < P; ++d) wa[d] = q24 * wa[d];
      }
    }
    const uint64_t m = __ballot(in);
    uint32_t slot = 0;
    if (m != 0ull) {
      const uint32_t leader = (uint32_t)__builtin_ctzll(m);
      if (lane == leader) slot = atomicAdd(&s_n, (uint32_t)__builtin_popcountll(m));
      slot = hmd_readlane(slot, leader) +
             (uint32_t)__builtin_popcountll(m & ((lane == 0) ? 0ull : (~0ull >> (64 - lane))));
    }
    if (in) {
#pragma unroll
      for (int d = 0; d < P; ++d) {
        s_w[0][d][slot] = wa[d];
        s_w[1][d][slot] = wb[d];
        s_w[2][d][slot] = wc[d];
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) s_at[d][slot] = (uint16_t)at[d];
    }
    __syncthreads();
    const uint32_t cnt = s_n;
    __syncthreads();   // every thread has the same count before it grows again
    // room for another round of candidates: go on collecting
    if (k0 + blockDim.x < total && cnt + blockDim.x <= Q) continue;
    for (uint32_t task = threadIdx.x; task < cnt * (uint32_t)P; task += blockDim.x) {
      const uint32_t e = task / (uint32_t)P, dc = task - e * (uint32_t)P;
      int lc = (int)s_at[2][e] - (int)dc;
      lc += (lc < 0) ? (int)p.n2 : 0;
      if (lc >= (int)p.b2) continue;
      const float w = s_w[2][dc][e];
      const int a0 = (int)s_at[0][e], b0 = (int)s_at[1][e];
      float wbv[P];
#pragma unroll
      for (int db = 0; db < P; ++db) wbv[db] = s_w[1][db][e];
#pragma unroll
      for (int da = 0; da < P; ++da) {
        int la = a0 - da;
        la += (la < 0) ? (int)p.n0 : 0;
        if (la >= (int)p.b0) continue;
        const float qa = s_w[0][da][e];
        long long* plane = s_acc + (uint32_t)la * p.b1 * p.b2 + (uint32_t)lc;
#pragma unroll
        for (int db = 0; db < P; ++db) {
          int lb = b0 - db;
          lb += (lb < 0) ? (int)p.n1 : 0;
          if (lb >= (int)p.b1) continue;
          atomicAdd(reinterpret_cast<unsigned long long*>(&plane[(uint32_t)lb * p.b2]),
                    (unsigned long long)hmd_fixed32_of24((qa * wbv[db]) * w));
        }
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
  }
  const float ib2 = 1.0f / (float)p.b2, ib1 = 1.0f / (float)p.b1;
  for (uint32_t k = threadIdx.x; k < bsz; k += blockDim.x) {
    const uint32_t row = hmd_div_small(k, ib2), lc = k - row * p.b2;
    const uint32_t la = hmd_div_small(row, ib1), lb = row - la * p.b1;
    const size_t gi = ((size_t)(o0 + la) * p.n1 + (o1 + lb)) * p.n2 + (o2 + lc);
    p.rho[gi] = hmd_from_fixed(s_acc[k], HMD_SPREAD_SHIFT);
  }
}

// The solve's reciprocal virial and energy (x, y) from its partials, summed in
// FP64 in a fixed order by a workgroup of 256: W = 0.5 sum hw vf |rho|^2,
// U = 0.5 sum hw G |rho|^2 (kernels/spme_recip.cu:376-402).
__device__ inline double2 hmd_spme_totals(const double* partials, uint32_t n) {
  __shared__ double2 s_part[4];
  double2 t = make_double2(0.0, 0.0);
  for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) {
    t.x += partials[2 * k];
    t.y += partials[2 * k + 1];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    t.x += __shfl_xor(t.x, o, HMD_WAVE);
    t.y += __shfl_xor(t.y, o, HMD_WAVE);
  }
  if (hmd_lane() == 0) s_part[threadIdx.x / HMD_WAVE] = t;
  __syncthreads();
  t.x = 0.5 * ((s_part[0].x + s_part[1].x) + (s_part[2].x + s_part[3].x));
  t.y = 0.5 * ((s_part[0].y + s_part[1].y) + (s_part[2].y + s_part[3].y));
  return t;
}

// The totals in a launch of their own, where the gather's workgroups would
// read too much for it (kSpmeSumInGather).
__device__ __forceinline__ void hmd_spme_reduce_body(const SpmeReduceParams& p,
                                                     const uint32_t hmd_bx,
                                                     const uint32_t hmd_gx) {
  const double2 t = hmd_spme_totals(p.partials, p.n_partials);
  if (threadIdx.x == 0) *reinterpret_cast<double2*>(p.totals) = t;
}
HMD_KERNEL(hmd_spme_reduce, SpmeReduceParams, 256)

// The partials of the solve are summed by every workgroup that hands the
// virial out (and by the first, which keeps the totals) while there are few:
// hmd_spme_reduce costs a launch.
template <int P>
__device__ inline void hmd_gather_body(const SpmeGatherParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  extern __shared__ float s_v[];
  const uint32_t h0 = p.b0 + P - 1, h1 = p.b1 + P - 1, h2 = p.b2 + P - 1;
  const uint32_t B = hmd_bx;
  const uint32_t B2 = B % p.nb2, B1 = (B / p.nb2) % p.nb1, B0 = B / (p.nb2 * p.nb1);
  const int o0 = (int)(B0 * p.b0) - (P - 1);
  const int o1 = (int)(B1 * p.b1) - (P - 1);
  const int o2 = (int)(B2 * p.b2) - (P - 1);
  double2 tot = make_double2(0.0, 0.0);
  if (p.n_partials == 0) {
    if (p.fev) tot = *reinterpret_cast<const double2*>(p.totals);
  } else if (p.fev || hmd_bx == 0) {
    tot = hmd_spme_totals(p.partials, p.n_partials);
    if (hmd_bx == 0 && threadIdx.x == 0) *reinterpret_cast<double2*>(p.totals) = tot;
  }
  const float ih2 = 1.0f / (float)h2, ih1 = 1.0f / (float)h1;
  for (uint32_t k = threadIdx.x; k < h0 * h1 * h2; k += blockDim.x) {
    const uint32_t row = hmd_div_small(k, ih2), lc = k - row * h2;
    const uint32_t la = hmd_div_small(row, ih1), lb = row - la * h1;
    int ga = o0 + (int)la, gb = o1 + (int)lb, gc = o2 + (int)lc;
    ga += ga < 0 ? (int)p.n0 : 0;
    gb += gb < 0 ? (int)p.n1 : 0;
    gc += gc < 0 ? (int)p.n2 : 0;
    s_v[k] = p.V[((size_t)ga * p.n1 + gb) * p.n2 + gc];
  }
  __syncthreads();

  const HmdLattice L = p.L;
  // Rows of H^{-T} for the lower-triangular cell
  // (spme_spread_gather.cuh:128-148).
  const float ilx = 1.0f / L.lx, ily = 1.0f / L.ly, ilz = 1.0f / L.lz;
  const float ba_x = ilx, ba_y = -L.xy * ilx * ily,
              ba_z = (L.xy * L.yz - L.xz * L.ly) * ilx * ily * ilz;
  const float bb_y = ily, bb_z = -L.yz * ily * ilz;
  const float bc_z = ilz;
  const float w_share = (float)(tot.x / (double)p.n);

  const uint32_t beg = p.bin_start[B], end = p.bin_start[B + 1];
  for (uint32_t k = beg + threadIdx.x; k < end; k += blockDim.x) {
    const uint32_t a = p.bin_atoms[k];
    const float4 pq = reinterpret_cast<const float4*>(p.posq)[a];
    float t[3];
    int g[3];
    hmd_spme_setup(pq, L, p.n0, p.n1, p.n2, t, g);
    float wa[P], wb[P], wc[P], dwa[P], dwb[P], dwc[P];
    hmd_bspline_deriv<P>(t[0], wa, dwa);
    hmd_bspline_deriv<P>(t[1], wb, dwb);
    hmd_bspline_deriv<P>(t[2], wc, dwc);
    // local halo coordinates of the primary point
    const int la0 = g[0] - o0, lb0 = g[1] - o1, lc0 = g[2] - o2;
    float phi = 0.0f, gra = 0.0f, grb = 0.0f, grc = 0.0f;
#pragma unroll
    for (int da = 0; da < P; ++da) {
#pragma unroll
      for (int db = 0; db < P; ++db) {
        const float* row = &s_v[((uint32_t)(la0 - da) * h1 + (uint32_t)(lb0 - db)) * h2];
        float sv = 0.0f, sdc = 0.0f;
#pragma unroll
        for (int dc = 0; dc < P; ++dc) {
          const float v = row[lc0 - dc];
          sv += v * wc[dc];
          sdc += v * dwc[dc];
        }
        phi += wa[da] * wb[db] * sv;
        gra += dwa[da] * wb[db] * sv;
        grb += wa[da] * dwb[db] * sv;
        grc += wa[da] * wb[db] * sdc;
      }
    }
    const float ga = (float)p.n0 * gra, gb = (float)p.n1 * grb, gc = (float)p.n2 * grc;
    p.f[a] = -pq.w * (ga * ba_x);
    p.f[p.n + a] = -pq.w * (ga * ba_y + gb * bb_y);
    p.f[2 * p.n + a] = -pq.w * (ga * ba_z + gb * bb_z + gc * bc_z);
    if (p.fev) {
      p.e[a] = 0.5f * pq.w * phi - p.u_self[a];
      p.w[a] = w_share;
    }
  }
}

#define HMD_SPME_ORDER(P)                                                    \
  __device__ __forceinline__ void hmd_spme_spread_p##P##_body(              \
      const SpmeSpreadParams& p, const uint32_t hmd_bx, const uint32_t hmd_gx) { \
    hmd_spread_body<P>(p, hmd_bx, hmd_gx);                                   \
  }                                                                          \
  __device__ __forceinline__ void hmd_spme_gather_p##P##_body(              \
      const SpmeGatherParams& p, const uint32_t hmd_bx, const uint32_t hmd_gx) { \
    hmd_gather_body<P>(p, hmd_bx, hmd_gx);                                   \
  }                                                                          \
  HMD_KERNEL(hmd_spme_spread_p##P, SpmeSpreadParams, 256)                    \
  HMD_KERNEL(hmd_spme_gather_p##P, SpmeGatherParams, 256)

HMD_SPME_ORDER(4)
HMD_SPME_ORDER(5)
HMD_SPME_ORDER(6)
HMD_SPME_ORDER(8)
