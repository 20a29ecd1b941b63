// Learned coarse-mesh SPME correction on gfx950: per-atom radial charge
// descriptors, and the pair-scalar MLP (51 -> 64 -> 64 -> 1, SiLU) forward
// and backward passes on the bf16 matrix cores with f32 accumulation.
//
// There is no counterpart in the reference (it has no learned component).
// The model: s = r/r_nn, phi_k(s) = exp(-(15 s - k)^2 / 2) (k = 0..15),
// fc(s) = (1 + cos(pi s))/2; D_i = sum_j q_j phi(s_ij) fc(s_ij);
// x_ij = [phi, one-hot(species_i + species_j), D_i, D_j];
// g_ij = s_out fc(s_ij) (N(x_ij) + N(x_ji)) / 2; dF_i = sum_j g_ij r^_ij.
//
// Traversal: the force field's packed half list (the pair kernel's).  The
// network passes compact the in-range pairs of each entry into an LDS queue
// and evaluate them 32 pairs (64 rows: both orientations) at a time:
//  * layer 1 is Z1^T = W1 X^T and layer 2 Z2^T = W2 H1^T as chains of
//    v_mfma_f32_16x16x32_bf16 (A = weights, B = activations); each lane
//    reads its slices of X^T whole from the wave's LDS tables;
//  * the layer-1 result registers (hidden h = 16t + 4g + r of row 16m + l%16,
//    g = l/16) are exactly the layer-2 B operand once the hidden units are
//    taken in the order pi(32k + 8g + e) = 16(2k + e/4) + 4g + e%4, so the
//    packed W2 columns follow pi and the activations never leave registers;
//  * per-pair forces go to LDS i64 fixed-point accumulators for the entry's
//    64 i- and 64 j-atoms, flushed with global i64 atomics (order-free sums:
//    bit-reproducible);
//  * the backward pass recomputes the forward per batch, chains dH1^T =
//    W2^T dZ2^T the same way, and accumulates the weight gradients
//    dW = dZ^T (rows) x A (rows) on the matrix cores, the two operands
//    turned by the transposing LDS read; per-wave partials are summed in a fixed
//    order by hmd_nn_grad_reduce.
#include "hmd_device.h"
#include "nn_items.h"

typedef __bf16 hmd_bf16x8 __attribute__((ext_vector_type(8)));
typedef float hmd_f32x4 __attribute__((ext_vector_type(4)));

#define HMD_NN_FORCE_SHIFT 40
#define HMD_NN_LOG2E 1.4426950408889634f
#define HMD_NN_QCAP 544u    // 8 i-atoms x 64 lanes + the < 32 pairs carried over
#define HMD_NN_TSTRIDE 72u  // transpose buffer row stride (bf16), 144 B

__device__ inline hmd_f32x4 hmd_mfma16(hmd_bf16x8 a, hmd_bf16x8 b, hmd_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ inline float hmd_sigmoid(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-z * HMD_NN_LOG2E));
}

__device__ inline void hmd_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ inline uint16_t hmd_bf16_bits(float v) {
  const __bf16 b = (__bf16)v;
  return __builtin_bit_cast(uint16_t, b);
}

typedef uint32_t hmd_u32x4 __attribute__((ext_vector_type(4)));

// Internal input order of the 64 (51 used) network inputs: rbf 0..15, one-hot
// 16..18, the first atom's descriptor 32..47, the second's 48..63.  The first
// half (one k-step of the matrix instruction) is the same for both
// orientations of a pair.  Returns the canonical index (rbf 0..15, one-hot
// 16..18, D_first 19..34, D_second 35..50) or -1 for padding.
__device__ inline int hmd_nn_canon_of_internal(uint32_t f) {
  if (f < 19u) return (int)f;
  if (f < 32u) return -1;
  return (int)(f - 13u);
}

// Hidden-unit order of the chained layer: B-operand k-index -> hidden unit.
__device__ inline uint32_t hmd_nn_pi(uint32_t k) {
  const uint32_t kap = k >> 5, g = (k >> 3) & 3u, e = k & 7u;
  return 16u * (2u * kap + (e >> 2)) + 4u * g + (e & 3u);
}

__device__ inline float hmd_nn_cutoff(float s) {
  // cos(pi s) through the native cosine, whose argument is in revolutions
  return 0.5f * (1.0f + __builtin_amdgcn_cosf(0.5f * s));
}

// phi_{k0 + e}(x), e = 0..7, for x = 15 s, by the Gaussian product
// recurrence phi_{k+1} = phi_k exp(x - k - 1/2), whose ratio itself shrinks
// by e^-1 per step: two exponentials instead of eight.  From k0 = 0 the
// start value underflows for x > 13.2, where phi_0..7 are below 6e-9; from
// k0 = 8 it never does.
__device__ inline void hmd_nn_rbf8(float u15, float k0, float out[8]) {
  const float t = u15 - k0;
  float ph = __builtin_amdgcn_exp2f(-0.5f * HMD_NN_LOG2E * t * t);
  float r = __builtin_amdgcn_exp2f(HMD_NN_LOG2E * (t - 0.5f));
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    out[e] = ph;
    ph *= r;
    r *= 0.36787944117144233f;
  }
}

__device__ inline uint32_t hmd_nn_species(uint32_t mask, uint32_t type) {
  return (mask >> (type & 31u)) & 1u;
}

// ---------------------------------------------------------- packing -----
// One thread per bf16 operand element (3 sets x 4 x 2 x 64 x 8).
extern "C" __global__ void __launch_bounds__(256)
hmd_nn_pack(const NnPackParams p) {
  const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
  const float* W1 = p.master;
  const float* b1 = W1 + 64 * 51;
  const float* W2 = b1 + 64;
  const float* b2 = W2 + 64 * 64;
  const float* w3 = b2 + 64;
  const float* b3 = w3 + 64;
  if (tid < 3u * 4u * 2u * 64u * 8u) {
    const uint32_t e = tid & 7u, lane = (tid >> 3) & 63u, kap = (tid >> 9) & 1u;
    const uint32_t t = (tid >> 10) & 3u, set = tid >> 12;
    const uint32_t row = 16u * t + (lane & 15u);
    const uint32_t k = 32u * kap + 8u * (lane >> 4) + e;
    float v = 0.0f;
    if (set == 0u) {
      const int cin = hmd_nn_canon_of_internal(k);
      v = cin >= 0 ? W1[row * 51u + (uint32_t)cin] : 0.0f;
    } else if (set == 1u) {
      v = W2[row * 64u + hmd_nn_pi(k)];
    } else {
      v = W2[hmd_nn_pi(k) * 64u + row];
    }
    p.ops[tid] = hmd_bf16_bits(v);
  }
  if (tid < 64u) {
    p.vec[tid] = b1[tid];
    p.vec[64 + tid] = b2[tid];
    p.vec[128 + tid] = (float)(__bf16)w3[tid];
  }
  if (tid == 0u) p.vec[192] = b3[0];
}

// Single-image shift of a cluster (compare jit_composed.rs:1396-1430, as in
// the pair kernel): valid when every atom within r_cut + r_skin/2 of the
// cluster lies within half a box of its centre; positions are then moved to
// the image nearest the centre and pair differences need no minimum image.
struct HmdNnShift {
  bool on;
  float cx, cy, cz;
};

__device__ inline HmdNnShift hmd_nn_cluster_shift(const NnPassParams& p, uint32_t c) {
  const HmdLattice& L = p.L;
  HmdNnShift sh{false, 0.0f, 0.0f, 0.0f};
  if (L.xy != 0.0f || L.xz != 0.0f || L.yz != 0.0f) return sh;
  const float4* bb = reinterpret_cast<const float4*>(p.bbox);
  const float4 cb = bb[2 * c], hb = bb[2 * c + 1];
  sh.on = (hb.x + p.shift_margin < 0.5f * L.lx) && (hb.y + p.shift_margin < 0.5f * L.ly) &&
          (hb.z + p.shift_margin < 0.5f * L.lz);
  sh.cx = cb.x; sh.cy = cb.y; sh.cz = cb.z;
  return sh;
}

__device__ inline float4 hmd_nn_apply_shift(float4 a, const HmdNnShift& sh, const HmdLattice& L) {
  if (sh.on) {
    a.x -= L.lx * floorf((a.x - sh.cx) * (1.0f / L.lx) + 0.5f);
    a.y -= L.ly * floorf((a.y - sh.cy) * (1.0f / L.ly) + 0.5f);
    a.z -= L.lz * floorf((a.z - sh.cz) * (1.0f / L.lz) + 0.5f);
  }
  return a;
}

// ------------------------------------------------------- descriptors ----
// The pair kernel's traversal: lane = j-atom of the entry (shifted once to
// the image nearest the i-cluster's centre), the i-atoms broadcast from an LDS
// table one per step, over the 8-atom i-sub-clusters the entry's mask admits
// (and the wave's item holds).  Per pair the 16 basis values come from two exponentials each half (the
// product recurrence of hmd_nn_rbf8) with the cutoff folded into their
// start; the j-atom's sums stay in the lane for the whole entry; the
// i-atom's 16 sums of the step are reduced over the wave by two transposed
// butterflies (totals of component m and 8 + m in lane 8m + 7) and added to
// the wave's i accumulators in LDS.  Sums go to i64 fixed point (2^32): the
// j side per entry, the i side per cluster share of the wave.
extern "C" __global__ void __launch_bounds__(64)
hmd_nn_descriptors(const NnPassParams p) {
#pragma clang fp contract(off)
  __shared__ float4 s_ip[HMD_CLUSTER];
  // i accumulators, component k of atom l at k * 65 + l (the odd stride
  // keeps the 8 lanes that add one atom's components on different banks)
  __shared__ float di[16 * 65];
  const uint32_t lane = threadIdx.x;
#pragma unroll
  for (int k = 0; k < 16; ++k) di[k * 65 + lane] = 0.0f;
  const uint32_t n_waves = gridDim.x, gw = blockIdx.x;
  const HmdNnItems items(__builtin_amdgcn_readfirstlane(*p.n_work), HMD_NN_ITEMS);
  if (gw >= items.n) return;
  const float4* ps = reinterpret_cast<const float4*>(p.posq_sorted);
  const HmdLattice L = p.L;
  long long* acc = p.desc_acc;
  const uint32_t stride = p.n_pad;

  uint32_t cur_c = HMD_SENTINEL, si = 0;
  bool vi = false;
  HmdNnShift sh{false, 0.0f, 0.0f, 0.0f};
  auto flush_i = [&]() {
    hmd_wave_sync();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const float v = di[k * 65 + lane];
      di[k * 65 + lane] = 0.0f;
      if (vi) hmd_atomic_add_fixed(&acc[k * stride + si], hmd_to_fixed(v, HMD_NN_DESC_SHIFT));
    }
  };
  for (uint32_t w = gw; w < items.n; w += n_waves) {
    const uint32_t slot = __builtin_amdgcn_readfirstlane(p.work[items.entry(w)]);
    uint32_t pend = __builtin_amdgcn_readfirstlane(p.entry_mask[slot]) & items.mask(w, n_waves);
    if (pend == 0u) continue;
    const uint32_t c = slot / p.cap_entries;
    const uint32_t c0 = c * HMD_CLUSTER;
    if (c != cur_c) {
      if (cur_c != HMD_SENTINEL) flush_i();
      cur_c = c;
      si = c0 + lane;
      vi = si < p.n;
      sh = hmd_nn_cluster_shift(p, c);
      float4 a = hmd_nn_apply_shift(ps[si], sh, L);
      if (!vi) a.x = a.y = a.z = 1.0e18f;   // padding lanes fail every cutoff test
      hmd_wave_sync();
      s_ip[lane] = a;
      hmd_wave_sync();
    }
    const uint32_t my_j = p.entry_j[(size_t)slot * HMD_ENTRY + lane];
    const bool valid_j = my_j != HMD_SENTINEL;
    float4 pj = hmd_nn_apply_shift(ps[valid_j ? my_j : 0u], sh, L);
    if (!valid_j) pj.x = pj.y = pj.z = 1.0e18f;
    // entries whose j-atoms all lie in later clusters need only the cutoff
    // test (i < j holds); the cluster's own entry also needs i < j
    const bool later = __ballot(valid_j && my_j < c0 + HMD_CLUSTER) == 0ull;
    float dj[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) dj[k] = 0.0f;
    while (pend) {
      const uint32_t sb = (uint32_t)__builtin_ctz(pend);
      pend &= pend - 1u;
#pragma unroll 2
      for (uint32_t u = 0; u < 8; ++u) {
        const uint32_t i = 8u * sb + u;
        const float4 a = s_ip[i];
        float dx = a.x - pj.x, dy = a.y - pj.y, dz = a.z - pj.z;
        if (!sh.on) hmd_min_image(dx, dy, dz, L);
        const float r2 = dx * dx + dy * dy + dz * dz;
        const bool ok = (r2 < p.r_cut2) && (r2 > 0.0f) && (later || c0 + i < my_j);
        if (__ballot(ok) == 0ull) continue;
        const float s = __builtin_sqrtf(ok ? r2 : 0.0f) * p.inv_r_cut;
        const float fc = ok ? hmd_nn_cutoff(s) : 0.0f;
        float w[16];
        hmd_nn_rbf8(15.0f * s, 0.0f, w);
        hmd_nn_rbf8(15.0f * s, 8.0f, w + 8);
        float vlo[8], vhi[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float wl = w[k] * fc, wh = w[8 + k] * fc;
          dj[k] = fmaf(a.w, wl, dj[k]);
          dj[8 + k] = fmaf(a.w, wh, dj[8 + k]);
          vlo[k] = pj.w * wl;
          vhi[k] = pj.w * wh;
        }
        const float tlo = hmd_wave_sum8(vlo, lane), thi = hmd_wave_sum8(vhi, lane);
        if ((lane & 7u) == 7u) {
          const uint32_t m = lane >> 3;
          di[m * 65 + i] += tlo;          // one lane per address: program order
          di[(8u + m) * 65 + i] += thi;
        }
      }
    }
    if (valid_j) {
#pragma unroll
      for (int k = 0; k < 16; ++k)
        hmd_atomic_add_fixed(&acc[k * stride + my_j], hmd_to_fixed(dj[k], HMD_NN_DESC_SHIFT));
    }
  }
  flush_i();
}

// Fixed point -> bf16 network inputs in sorted order (and f32 descriptors in
// canonical order when asked); the accumulators are cleared for the next evaluation.
extern "C" __global__ void __launch_bounds__(256)
hmd_nn_desc_finalize(const NnDescFinalizeParams p) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= p.n_pad) return;
  const uint32_t id = p.sorted_id[s];
  hmd_bf16x8 d[2];
#pragma unroll
  for (uint32_t k = 0; k < 16; ++k) {
    const float v = hmd_from_fixed(p.desc_acc[k * p.n_pad + s], HMD_NN_DESC_SHIFT);
    p.desc_acc[k * p.n_pad + s] = 0;
    d[k >> 3][k & 7u] = (__bf16)v;
    if (p.desc_canon && s < p.n) p.desc_canon[id * 16 + k] = v;
  }
  hmd_bf16x8* out = reinterpret_cast<hmd_bf16x8*>(p.desc) + 2 * (size_t)s;
  out[0] = d[0];
  out[1] = d[1];
}

// ------------------------------------------------ network passes --------
// Per-wave tables of the current entry: its i-atoms (0..63) and j-atoms
// (64..127), positions shifted to the image nearest the cluster centre when
// the cluster qualifies (w: species), their descriptors, and the queue of
// in-range pairs; then the 64 inputs' first half of a batch's pairs.
struct HmdNnTables {
  float4 pos[2 * HMD_WAVE];
  hmd_bf16x8 dsc[2 * HMD_WAVE][2];         // descriptors, bf16
  hmd_bf16x8 xin[32][4];                   // inputs 0..31: rbf, one-hot, zeros
  float4 geo[32];                          // fc, unit vector i - j
  uint16_t queue[HMD_NN_QCAP];             // (i lane) | (j slot << 6)
};

// Table row of an atom: position (w: species) and descriptors.
__device__ inline void hmd_nn_load_atom(const NnPassParams& p, HmdNnTables& W, uint32_t row,
                                        uint32_t s, float4 a) {
  a.w = (float)hmd_nn_species(p.species_mask, p.type_sorted[s]);
  W.pos[row] = a;
  const hmd_bf16x8* d = reinterpret_cast<const hmd_bf16x8*>(p.desc) + 2 * (size_t)s;
  W.dsc[row][0] = d[0];
  W.dsc[row][1] = d[1];
}

__device__ inline float4 hmd_nn_resid(const NnPassParams& p, uint32_t s) {
  return make_float4(p.resid[s], p.resid[p.n_pad + s], p.resid[2 * p.n_pad + s], 0.0f);
}

// Append the in-range pairs of i-sub-cluster sb to the wave queue: lane =
// j-atom, the eight i-atoms broadcast from the table.  j_lim is the lane's
// j-atom, 0 on lanes without one.
__device__ inline uint32_t hmd_nn_compact(const NnPassParams& p, HmdNnTables& W, uint32_t sb,
                                          uint32_t c0, uint32_t n_i, float4 pj, uint32_t j_lim,
                                          bool shift, uint32_t qn, uint32_t lane) {
#pragma unroll
  for (uint32_t u = 0; u < 8; ++u) {
    const uint32_t i = 8u * sb + u;
    const float4 a = W.pos[i];
    float dx = a.x - pj.x, dy = a.y - pj.y, dz = a.z - pj.z;
    if (!shift) hmd_min_image(dx, dy, dz, p.L);
    const float r2 = dx * dx + dy * dy + dz * dz;
    const bool ok = (r2 < p.r_cut2) && (r2 > 0.0f) && (c0 + i < j_lim) && (i < n_i);
    const uint64_t m = __ballot(ok);
    if (ok) {
      const uint32_t at = __builtin_amdgcn_mbcnt_hi(
          (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, qn));
      W.queue[at] = (uint16_t)(i | (lane << 6));
    }
    qn += (uint32_t)__builtin_popcountll(m);
  }
  return qn;
}

// Geometry and the first half of the inputs of the queue's pairs
// [base, base + 32): lanes l and l + 32 take pair l, each half of the basis.
// Slots past cnt hold a pair at unit distance with a zero cutoff factor.
__device__ inline void hmd_nn_pair_inputs(const NnPassParams& p, HmdNnTables& W, uint32_t base,
                                          uint32_t cnt, bool shift, uint32_t lane) {
  const uint32_t pr = lane & 31u, hf = lane >> 5;
  const bool valid = pr < cnt;
  const uint32_t q = valid ? W.queue[base + pr] : 0u;
  const float4 a = W.pos[q & 63u], b = W.pos[HMD_WAVE + (q >> 6)];
  float dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
  if (!shift) hmd_min_image(dx, dy, dz, p.L);
  const float r2 = valid ? dx * dx + dy * dy + dz * dz : 1.0f;
  const float inv_r = __builtin_amdgcn_rsqf(r2);
  const float sc = r2 * inv_r * p.inv_r_cut;
  float phf[8];
  hmd_nn_rbf8(15.0f * sc, (float)(8u * hf), phf);
  hmd_bf16x8 ph;
#pragma unroll
  for (int e = 0; e < 8; ++e) ph[e] = (__bf16)phf[e];
  W.xin[pr][hf] = ph;
  if (hf == 0u) {
    const float fc = valid ? hmd_nn_cutoff(sc) : 0.0f;
    W.geo[pr] = make_float4(fc, dx * inv_r, dy * inv_r, dz * inv_r);
  } else {
    const float oh = a.w + b.w;
    hmd_u32x4 w = {0u, 0u, 0u, 0u};
    w[0] = oh == 0.0f ? 0x3F80u : (oh == 1.0f ? 0x3F800000u : 0u);
    w[1] = oh == 2.0f ? 0x3F80u : 0u;
    W.xin[pr][2] = __builtin_bit_cast(hmd_bf16x8, w);
  }
}

// SiLU of the eight hidden units a lane holds of one row and one pair of
// tiles, as the next layer's operand.
__device__ inline hmd_bf16x8 hmd_nn_silu8(hmd_f32x4 a, hmd_f32x4 b) {
  hmd_bf16x8 h;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    h[r] = (__bf16)(a[r] * hmd_sigmoid(a[r]));
    h[4 + r] = (__bf16)(b[r] * hmd_sigmoid(b[r]));
  }
  return h;
}

// Weights of the forward pass, held in registers for the whole kernel.
struct HmdNnFwdRegs {
  hmd_bf16x8 w1[4][2], w2[4][2];
  hmd_f32x4 b1[4], b2[4], w3[4];
  float b3;
};

// Forward: dF into the fixed-point accumulators (sorted order).
//
// A batch is 32 pairs: its geometry and inputs go through a per-wave LDS
// table, then 16 pairs at a time run through the two layers in both
// orientations side by side.  The first k-step of layer 1 (basis and
// one-hot, bias as the accumulator's start) is shared by the orientations;
// two independent chains keep the transcendental unit fed while a matrix
// result is in flight.  Bound by the VALU: 128 SiLUs a lane and batch (an
// exponential and a reciprocal each).  Weights and biases stay in registers
// (two waves per SIMD) and results in architectural VGPRs; with weights in
// LDS, one tile in flight and the results moved out of the accumulation
// registers, 24,576 atoms took 1,585 us and 196,608 atoms 6.18 ms, then 1,216
// us and 4.64 ms.
__device__ inline void hmd_nn_forward_batch(const NnPassParams& p, const HmdNnFwdRegs& R,
                                            HmdNnTables& W, long long (*acc)[3][HMD_WAVE],
                                            uint32_t base, uint32_t cnt, bool shift,
                                            uint32_t lane) {
  const uint32_t g = lane >> 4, pl = lane & 15u;
  hmd_nn_pair_inputs(p, W, base, cnt, shift, lane);
  hmd_wave_sync();
  float y0 = 0.0f, y1 = 0.0f;
#pragma unroll 1
  for (uint32_t h = 0; 16u * h < cnt; ++h) {
    const uint32_t q = W.queue[base + 16u * h + pl];
    const uint32_t ri = q & 63u, rj = HMD_WAVE + ((q >> 6) & 63u);
    const hmd_bf16x8 x0 = W.xin[16u * h + pl][g];
    const hmd_bf16x8 xa = W.dsc[g < 2u ? ri : rj][g & 1u];
    const hmd_bf16x8 xb = W.dsc[g < 2u ? rj : ri][g & 1u];
    hmd_f32x4 za[4], zb[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const hmd_f32x4 c = hmd_mfma16(R.w1[t][0], x0, R.b1[t]);
      za[t] = hmd_mfma16(R.w1[t][1], xa, c);
      zb[t] = hmd_mfma16(R.w1[t][1], xb, c);
    }
    const hmd_bf16x8 ha0 = hmd_nn_silu8(za[0], za[1]), hb0 = hmd_nn_silu8(zb[0], zb[1]);
    const hmd_bf16x8 ha1 = hmd_nn_silu8(za[2], za[3]), hb1 = hmd_nn_silu8(zb[2], zb[3]);
    float ya = 0.0f, yb = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const hmd_f32x4 ca = hmd_mfma16(R.w2[t][1], ha1, hmd_mfma16(R.w2[t][0], ha0, R.b2[t]));
      const hmd_f32x4 cb = hmd_mfma16(R.w2[t][1], hb1, hmd_mfma16(R.w2[t][0], hb0, R.b2[t]));
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ya = fmaf(R.w3[t][r], ca[r] * hmd_sigmoid(ca[r]), ya);
        yb = fmaf(R.w3[t][r], cb[r] * hmd_sigmoid(cb[r]), yb);
      }
    }
    (h ? y1 : y0) = ya + yb;
  }
  y0 += hmd_shfl_xor(y0, 16);
  y1 += hmd_shfl_xor(y1, 16);
  y0 += hmd_shfl_xor(y0, 32);
  y1 += hmd_shfl_xor(y1, 32);
  // lane l < 32 applies pair l
  if (lane < cnt && lane < 32u) {
    const float4 geo = W.geo[lane];
    const float gp = p.force_scale * geo.x * 0.5f * ((g ? y1 : y0) + 2.0f * R.b3);
    const uint32_t q = W.queue[base + lane];
    const uint32_t ia = q & 63u, jk = q >> 6;
    const float rh[3] = {geo.y, geo.z, geo.w};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const long long f = hmd_to_fixed(gp * rh[d], HMD_NN_FORCE_SHIFT);
      atomicAdd(reinterpret_cast<unsigned long long*>(&acc[0][d][ia]),
                static_cast<unsigned long long>(f));
      atomicAdd(reinterpret_cast<unsigned long long*>(&acc[1][d][jk]),
                static_cast<unsigned long long>(-f));
    }
  }
  hmd_wave_sync();
}

// One wave a workgroup: nothing is shared between waves, and a workgroup of
// four held three idle SIMDs until its slowest wave was done (62% of the SIMDs
// had a wave on average): 24,576 atoms 1,000 -> 741 us a pass.
extern "C" __global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2)))
hmd_nn_forward(const NnPassParams p) {
  __shared__ HmdNnTables W;
  __shared__ long long acc[2][3][HMD_WAVE];
  const uint32_t lane = threadIdx.x;
  const uint32_t n_waves = gridDim.x, gw = blockIdx.x;
  const HmdNnItems items(__builtin_amdgcn_readfirstlane(*p.n_work), HMD_NN_ITEMS);
  if (gw >= items.n) return;
  const float4* ps = reinterpret_cast<const float4*>(p.posq_sorted);
  const uint32_t stride = p.n_pad;
  const uint32_t g = lane >> 4;
  HmdNnFwdRegs R;
  {
    const hmd_bf16x8* ops = reinterpret_cast<const hmd_bf16x8*>(p.ops);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        R.w1[t][k] = ops[(2 * t + k) * HMD_WAVE + lane];
        R.w2[t][k] = ops[(8 + 2 * t + k) * HMD_WAVE + lane];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        R.b1[t][r] = p.vec[16 * t + 4 * g + r];
        R.b2[t][r] = p.vec[64 + 16 * t + 4 * g + r];
        R.w3[t][r] = p.vec[128 + 16 * t + 4 * g + r];
      }
    }
    R.b3 = p.vec[192];
  }
  if (lane < 32u) W.xin[lane][3] = __builtin_bit_cast(hmd_bf16x8, hmd_u32x4{0u, 0u, 0u, 0u});
#pragma unroll
  for (int d = 0; d < 3; ++d) { acc[0][d][lane] = 0; acc[1][d][lane] = 0; }

  uint32_t cur_c = HMD_SENTINEL, si = 0, n_i = 0;
  bool vi = false;
  HmdNnShift sh{false, 0.0f, 0.0f, 0.0f};
  for (uint32_t w = gw; w < items.n; w += n_waves) {
    const uint32_t slot = __builtin_amdgcn_readfirstlane(p.work[items.entry(w)]);
    uint32_t pend = __builtin_amdgcn_readfirstlane(p.entry_mask[slot]) & items.mask(w, n_waves);
    if (pend == 0u) continue;
    const uint32_t c = slot / p.cap_entries;
    const uint32_t my_j = p.entry_j[(size_t)slot * HMD_ENTRY + lane];
    hmd_wave_sync();
    if (c != cur_c) {
      if (cur_c != HMD_SENTINEL) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const long long v = acc[0][d][lane];
          acc[0][d][lane] = 0;
          if (vi) hmd_atomic_add_fixed(&p.force_acc[d * stride + si], v);
        }
      }
      cur_c = c;
      si = c * HMD_CLUSTER + lane;
      vi = si < p.n;
      n_i = min((uint32_t)HMD_CLUSTER, p.n - c * HMD_CLUSTER);
      sh = hmd_nn_cluster_shift(p, c);
      hmd_nn_load_atom(p, W, lane, si, hmd_nn_apply_shift(ps[si], sh, p.L));
    }
    const bool valid_j = my_j != HMD_SENTINEL;
    const uint32_t jj = valid_j ? my_j : 0u;
    const float4 pj = hmd_nn_apply_shift(ps[jj], sh, p.L);
    hmd_nn_load_atom(p, W, HMD_WAVE + lane, jj, pj);
    hmd_wave_sync();
    uint32_t qn = 0;
    while (pend) {
      const uint32_t sb = (uint32_t)__builtin_ctz(pend);
      pend &= pend - 1u;
      qn = hmd_nn_compact(p, W, sb, c * HMD_CLUSTER, n_i, pj, jj, sh.on, qn, lane);
      hmd_wave_sync();
      // full batches now, the rest with the next sub-cluster or at the end
      const uint32_t keep = pend ? qn & 31u : 0u;
      uint32_t head = 0;
      for (; head + keep < qn; head += 32u)
        hmd_nn_forward_batch(p, R, W, acc, head, min(qn - head, 32u), sh.on, lane);
      if (keep && head) {
        const uint16_t carry = lane < keep ? W.queue[head + lane] : (uint16_t)0;
        hmd_wave_sync();
        if (lane < keep) W.queue[lane] = carry;
        hmd_wave_sync();
      }
      qn = keep;
    }
    hmd_wave_sync();
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const long long v = acc[1][d][lane];
      acc[1][d][lane] = 0;
      if (valid_j) hmd_atomic_add_fixed(&p.force_acc[d * stride + my_j], v);
    }
  }
  hmd_wave_sync();
  if (vi) {
#pragma unroll
    for (int d = 0; d < 3; ++d) hmd_atomic_add_fixed(&p.force_acc[d * stride + si], acc[0][d][lane]);
  }
}

// Backward: weight gradients of sum over rows of dy * y, with dy from the
// residual dL/d(dF) of the two atoms; per-wave partials.
struct HmdNnGrad {
  hmd_f32x4 w1[4][4], w2[4][4];    // [hidden tile][input tile]
  hmd_f32x4 b1[4], b2[4], w3[4];
  float b3;
};

struct HmdNnShared {
  hmd_bf16x8 ops[3][8][HMD_WAVE];          // W1, W2, W2^T operands
  float vec[HMD_NN_HID * 3 + 4];           // b1, b2, w3, b3
};

struct HmdNnWave : HmdNnTables {
  float4 res[2 * HMD_WAVE];                // dL/d(dF) of the table's atoms
  // rows (16 pairs, both orientations) x 64 columns of the two factors of a
  // weight gradient
  __attribute__((aligned(16))) uint16_t T[2][32][HMD_NN_TSTRIDE];
};

__device__ inline void hmd_nn_load_shared(const NnPassParams& p, HmdNnShared& S) {
  const hmd_bf16x8* ops = reinterpret_cast<const hmd_bf16x8*>(p.ops);
  for (uint32_t k = threadIdx.x; k < 24u * HMD_WAVE; k += blockDim.x)
    (&S.ops[0][0][0])[k] = ops[k];
  for (uint32_t k = threadIdx.x; k < HMD_NN_HID * 3 + 1; k += blockDim.x) S.vec[k] = p.vec[k];
  __syncthreads();
}

typedef short hmd_s16x4 __attribute__((ext_vector_type(4)));

// Column 16 t + l % 16 of a row-major [32][64] table as a matrix operand
// whose k index runs over the rows: two transposing LDS reads, each giving
// the lanes of a group of 16 the 16 columns of 4 rows (8 g + 4 j ..).
__device__ inline hmd_bf16x8 hmd_nn_column(const uint16_t (*T)[HMD_NN_TSTRIDE], int t,
                                           uint32_t lane) {
  typedef __attribute__((address_space(3))) hmd_s16x4* lds_ptr;
  const uint32_t row = 8u * (lane >> 4) + ((lane & 15u) >> 2), col = 16u * t + 4u * (lane & 3u);
  const hmd_s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)&T[row][col]);
  const hmd_s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)&T[row + 4u][col]);
  return __builtin_bit_cast(hmd_bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// The four hidden units 16 t + 4 g .. of a row, into its table row.
__device__ inline void hmd_nn_put4(uint16_t* row, uint32_t t, uint32_t g, hmd_bf16x8 v, int half) {
  const hmd_u32x4 w = __builtin_bit_cast(hmd_u32x4, v);
  *reinterpret_cast<uint2*>(row + 16u * t + 4u * g) =
      half ? make_uint2(w[2], w[3]) : make_uint2(w[0], w[1]);
}

// SiLU of four units: values to out, derivatives returned.
__device__ inline hmd_f32x4 hmd_nn_silu_d(hmd_f32x4 z, float out[4]) {
  hmd_f32x4 d;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float s = hmd_sigmoid(z[r]);
    const float h = z[r] * s;
    out[r] = h;
    d[r] = fmaf(h, 1.0f - s, s);      // s (1 + z (1 - s))
  }
  return d;
}

// 16 pairs = 32 rows, the contraction length of one matrix instruction of
// the weight gradients.  The activations stay in the layer-chaining layout
// (lane = row); the factors of a weight gradient need lane = unit, which the
// transposing LDS read gives from rows written four units at a time.  One
// wave per SIMD: the 176 registers of gradient sums and two rows' activations
// fit without spills (64 rows at a time spilled 652 B a lane and transposed
// by 256 two-byte LDS writes): 9,999 atoms 2,452 -> 1,427 us.
__device__ inline void hmd_nn_backward_rows(const NnPassParams& p, const HmdNnShared& S,
                                            HmdNnWave& W, HmdNnGrad& G, uint32_t q, uint32_t pr,
                                            uint32_t lane) {
  const uint32_t g = lane >> 4, pl = lane & 15u;
  const uint32_t ri = q & 63u, rj = HMD_WAVE + ((q >> 6) & 63u);
  const hmd_bf16x8 x0 = W.xin[pr][g];
  const hmd_bf16x8 xa = W.dsc[g < 2u ? ri : rj][g & 1u];
  const hmd_bf16x8 xb = W.dsc[g < 2u ? rj : ri][g & 1u];
  const float4 geo = W.geo[pr], fi = W.res[ri], fj = W.res[rj];
  const float dg = (fi.x - fj.x) * geo.y + (fi.y - fj.y) * geo.z + (fi.z - fj.z) * geo.w;
  const float dy = dg * p.force_scale * geo.x * 0.5f;   // geo.x = 0 on unused rows
  if (g == 0u) G.b3 += 2.0f * dy;
  const hmd_f32x4* b1 = reinterpret_cast<const hmd_f32x4*>(S.vec) + g;
  const hmd_f32x4* b2 = b1 + 16;
  const hmd_f32x4* w3 = b1 + 32;
  uint16_t (*T0)[HMD_NN_TSTRIDE] = W.T[0];
  uint16_t (*T1)[HMD_NN_TSTRIDE] = W.T[1];

  hmd_f32x4 da[4], db[4];
  hmd_bf16x8 ha[2], hb[2];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const hmd_f32x4 c = hmd_mfma16(S.ops[0][2 * t][lane], x0, b1[4 * t]);
    const hmd_bf16x8 w = S.ops[0][2 * t + 1][lane];
    float va[4], vb[4];
    da[t] = hmd_nn_silu_d(hmd_mfma16(w, xa, c), va);
    db[t] = hmd_nn_silu_d(hmd_mfma16(w, xb, c), vb);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ha[t >> 1][4 * (t & 1) + r] = (__bf16)va[r];
      hb[t >> 1][4 * (t & 1) + r] = (__bf16)vb[r];
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    hmd_nn_put4(T1[pl], t, g, ha[t >> 1], t & 1);
    hmd_nn_put4(T1[16u + pl], t, g, hb[t >> 1], t & 1);
  }
  // output layer and layer-2 error signal
  hmd_bf16x8 ea[2], eb[2];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const hmd_bf16x8 w0 = S.ops[1][2 * t][lane], w1 = S.ops[1][2 * t + 1][lane];
    const hmd_f32x4 c = b2[4 * t], w = w3[4 * t];
    float va[4], vb[4];
    const hmd_f32x4 sa = hmd_nn_silu_d(hmd_mfma16(w1, ha[1], hmd_mfma16(w0, ha[0], c)), va);
    const hmd_f32x4 sb = hmd_nn_silu_d(hmd_mfma16(w1, hb[1], hmd_mfma16(w0, hb[0], c)), vb);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      G.w3[t][r] = fmaf(dy, va[r] + vb[r], G.w3[t][r]);
      const float wd = w[r] * dy;
      const float za = wd * sa[r], zb = wd * sb[r];
      G.b2[t][r] += za + zb;
      ea[t >> 1][4 * (t & 1) + r] = (__bf16)za;
      eb[t >> 1][4 * (t & 1) + r] = (__bf16)zb;
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    hmd_nn_put4(T0[pl], t, g, ea[t >> 1], t & 1);
    hmd_nn_put4(T0[16u + pl], t, g, eb[t >> 1], t & 1);
  }
  hmd_wave_sync();
  // dW2 += dZ2^T H1 over the 32 rows
  {
    hmd_bf16x8 b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) b[t] = hmd_nn_column(T1, t, lane);
#pragma unroll
    for (int to = 0; to < 4; ++to) {
      const hmd_bf16x8 a = hmd_nn_column(T0, to, lane);
#pragma unroll
      for (int ti = 0; ti < 4; ++ti) G.w2[to][ti] = hmd_mfma16(a, b[ti], G.w2[to][ti]);
    }
  }
  hmd_wave_sync();
  // dH1^T = W2^T dZ2^T (chained), layer-1 error signal
  hmd_bf16x8 za[2], zb[2];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const hmd_bf16x8 w0 = S.ops[2][2 * t][lane], w1 = S.ops[2][2 * t + 1][lane];
    const hmd_f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const hmd_f32x4 ca = hmd_mfma16(w1, ea[1], hmd_mfma16(w0, ea[0], zero));
    const hmd_f32x4 cb = hmd_mfma16(w1, eb[1], hmd_mfma16(w0, eb[0], zero));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float a = ca[r] * da[t][r], b = cb[r] * db[t][r];
      G.b1[t][r] += a + b;
      za[t >> 1][4 * (t & 1) + r] = (__bf16)a;
      zb[t >> 1][4 * (t & 1) + r] = (__bf16)b;
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    hmd_nn_put4(T0[pl], t, g, za[t >> 1], t & 1);
    hmd_nn_put4(T0[16u + pl], t, g, zb[t >> 1], t & 1);
  }
  *reinterpret_cast<hmd_bf16x8*>(&T1[pl][8u * g]) = x0;
  *reinterpret_cast<hmd_bf16x8*>(&T1[pl][32u + 8u * g]) = xa;
  *reinterpret_cast<hmd_bf16x8*>(&T1[16u + pl][8u * g]) = x0;
  *reinterpret_cast<hmd_bf16x8*>(&T1[16u + pl][32u + 8u * g]) = xb;
  hmd_wave_sync();
  // dW1 += dZ1^T X over the rows
  {
    hmd_bf16x8 b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) b[t] = hmd_nn_column(T1, t, lane);
#pragma unroll
    for (int th = 0; th < 4; ++th) {
      const hmd_bf16x8 a = hmd_nn_column(T0, th, lane);
#pragma unroll
      for (int tf = 0; tf < 4; ++tf) G.w1[th][tf] = hmd_mfma16(a, b[tf], G.w1[th][tf]);
    }
  }
  hmd_wave_sync();
}

extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
hmd_nn_backward(const NnPassParams p) {
  __shared__ HmdNnShared S;
  __shared__ HmdNnWave Wv[4];
  hmd_nn_load_shared(p, S);
  const uint32_t lane = hmd_lane();
  const uint32_t wv = threadIdx.x / HMD_WAVE;
  const uint32_t n_waves = gridDim.x * (blockDim.x / HMD_WAVE);
  const uint32_t gw = blockIdx.x * (blockDim.x / HMD_WAVE) + wv;
  const HmdNnItems items(__builtin_amdgcn_readfirstlane(*p.n_work), HMD_NN_ITEMS);
  HmdNnWave& W = Wv[wv];
  const float4* ps = reinterpret_cast<const float4*>(p.posq_sorted);
  if (lane < 32u) W.xin[lane][3] = __builtin_bit_cast(hmd_bf16x8, hmd_u32x4{0u, 0u, 0u, 0u});

  HmdNnGrad G;
  const hmd_f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int a = 0; a < 4; ++a) {
#pragma unroll
    for (int b = 0; b < 4; ++b) G.w1[a][b] = G.w2[a][b] = zero;
    G.b1[a] = G.b2[a] = G.w3[a] = zero;
  }
  G.b3 = 0.0f;

  uint32_t cur_c = HMD_SENTINEL, n_i = 0;
  HmdNnShift sh{false, 0.0f, 0.0f, 0.0f};
  for (uint32_t w = gw; w < items.n; w += n_waves) {
    const uint32_t slot = __builtin_amdgcn_readfirstlane(p.work[items.entry(w)]);
    uint32_t pend = __builtin_amdgcn_readfirstlane(p.entry_mask[slot]) & items.mask(w, n_waves);
    if (pend == 0u) continue;
    const uint32_t c = slot / p.cap_entries;
    const uint32_t my_j = p.entry_j[(size_t)slot * HMD_ENTRY + lane];
    hmd_wave_sync();
    if (c != cur_c) {
      cur_c = c;
      const uint32_t si = c * HMD_CLUSTER + lane;
      n_i = min((uint32_t)HMD_CLUSTER, p.n - c * HMD_CLUSTER);
      sh = hmd_nn_cluster_shift(p, c);
      hmd_nn_load_atom(p, W, lane, si, hmd_nn_apply_shift(ps[si], sh, p.L));
      W.res[lane] = hmd_nn_resid(p, si);
    }
    const uint32_t jj = my_j != HMD_SENTINEL ? my_j : 0u;
    const float4 pj = hmd_nn_apply_shift(ps[jj], sh, p.L);
    hmd_nn_load_atom(p, W, HMD_WAVE + lane, jj, pj);
    W.res[HMD_WAVE + lane] = hmd_nn_resid(p, jj);
    hmd_wave_sync();
    uint32_t qn = 0;
    while (pend) {
      const uint32_t sb = (uint32_t)__builtin_ctz(pend);
      pend &= pend - 1u;
      qn = hmd_nn_compact(p, W, sb, c * HMD_CLUSTER, n_i, pj, jj, sh.on, qn, lane);
      hmd_wave_sync();
      const uint32_t keep = pend ? qn & 31u : 0u;
      uint32_t head = 0;
      for (; head + keep < qn; head += 32u) {
        const uint32_t cnt = min(qn - head, 32u);
        hmd_nn_pair_inputs(p, W, head, cnt, sh.on, lane);
        hmd_wave_sync();
#pragma unroll 1
        for (uint32_t pr = 0; pr < cnt; pr += 16u) {
          const uint32_t at = pr + (lane & 15u);
          const uint32_t q = at < cnt ? W.queue[head + at] : 0u;
          hmd_nn_backward_rows(p, S, W, G, q, at, lane);
        }
      }
      if (keep && head) {
        const uint16_t carry = lane < keep ? W.queue[head + lane] : (uint16_t)0;
        hmd_wave_sync();
        if (lane < keep) W.queue[lane] = carry;
        hmd_wave_sync();
      }
      qn = keep;
    }
  }

  float* out = p.partials + (size_t)gw * HMD_NN_PARTIAL;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        out[((a * 4 + b) * 4 + r) * 64 + lane] = G.w1[a][b][r];
        out[4096 + ((a * 4 + b) * 4 + r) * 64 + lane] = G.w2[a][b][r];
      }
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      out[8192 + (t * 4 + r) * 64 + lane] = G.b1[t][r];
      out[9216 + (t * 4 + r) * 64 + lane] = G.b2[t][r];
      out[10240 + (t * 4 + r) * 64 + lane] = G.w3[t][r];
    }
  out[11264 + lane] = G.b3;
}

// Canonical gradient from the per-wave partials: one workgroup per 64-float
// row of the partials (177 rows), its 16 waves taking backward waves w =
// v, v + 16, ... (coalesced 256-byte reads), then the 16 sums and, for the
// bias rows, the lanes of a parameter in increasing order: FP64, a fixed
// summation order.  One workgroup per parameter read 4 bytes of every
// partial: 83 us, now 9.7 us (46 MB).
extern "C" __global__ void __launch_bounds__(1024)
hmd_nn_grad_reduce(const NnGradReduceParams p) {
  __shared__ double s_sum[16][HMD_WAVE];
  const uint32_t row = blockIdx.x, lane = hmd_lane(), wv = threadIdx.x / HMD_WAVE;
  double acc = 0.0;
#pragma unroll 8
  for (uint32_t w = wv; w < p.n_waves; w += 16u)
    acc += (double)p.partials[(size_t)w * HMD_NN_PARTIAL + row * HMD_WAVE + lane];
  s_sum[wv][lane] = acc;
  __syncthreads();
  if (wv != 0u) return;
  acc = 0.0;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc += s_sum[v][lane];
  const uint32_t W2 = 64u * 51u + 64u, g = lane >> 4;
  if (row < 128u) {                                      // W1[h][cin], W2[h][f]
    const uint32_t h = 16u * ((row >> 4) & 3u) + 4u * g + (row & 3u);
    const uint32_t f = 16u * ((row >> 2) & 3u) + (lane & 15u);
    if (row < 64u) {
      const int cin = hmd_nn_canon_of_internal(f);
      if (cin >= 0) p.grad[h * 51u + (uint32_t)cin] += acc;
    } else {
      p.grad[W2 + h * 64u + f] += acc;
    }
    return;
  }
  s_sum[0][lane] = acc;
  hmd_wave_sync();
  if (row == 176u) {                                     // b3
    if (lane == 0u) {
      double s = 0.0;
      for (int l = 0; l < 64; ++l) s += s_sum[0][l];
      p.grad[W2 + 4096u + 128u] += s;
    }
  } else if ((lane & 15u) == 0u) {                       // b1, b2, w3 [h]
    const uint32_t set = (row - 128u) >> 4, tr = (row - 128u) & 15u;
    const uint32_t h = 16u * (tr >> 2) + 4u * g + (tr & 3u);
    double s = 0.0;
    for (uint32_t l = 0; l < 16u; ++l) s += s_sum[0][lane + l];
    p.grad[(set == 0u ? 64u * 51u : W2 + 4096u + 64u * (set - 1u)) + h] += s;
  }
}

// ------------------------------------------------------------ helpers ---
extern "C" __global__ void __launch_bounds__(256)
hmd_nn_finalize(const NnFinalizeParams p) {
  const uint32_t a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= p.n) return;
  const uint32_t s = p.slot_of[a];
#pragma unroll
  for (uint32_t d = 0; d < 3; ++d) {
    const float v = hmd_from_fixed(p.force_acc[d * p.n_pad + s], HMD_NN_FORCE_SHIFT);
    p.force_acc[d * p.n_pad + s] = 0;
    p.df[d * p.n + a] = v;
    if (p.add_to) p.add_to[d * p.n + a] += v;
  }
}

extern "C" __global__ void __launch_bounds__(256)
hmd_nn_residual(const NnResidualParams p) {
  __shared__ double s[256];
  const uint32_t a = blockIdx.x * blockDim.x + threadIdx.x;
  double acc = 0.0;
  if (a < p.n) {
    const uint32_t slot = p.slot_of[a];
#pragma unroll
    for (uint32_t d = 0; d < 3; ++d) {
      const float r = p.df[d * p.n + a] - p.target[d * p.n + a];
      p.resid[d * p.n_pad + slot] = p.scale * r;
      acc += (double)r * (double)r;
    }
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (uint32_t st = blockDim.x / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) s[threadIdx.x] += s[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) p.partials[blockIdx.x] = s[0] * p.loss_scale;
}

// Adam (Kingma & Ba 2015, Algorithm 1) on the f32 master copy; the
// accumulated FP64 gradient is cleared.
extern "C" __global__ void __launch_bounds__(256)
hmd_nn_adam(const NnAdamParams p) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= HMD_NN_PARAMS) return;
  const float g = (float)p.grad[k];
  p.grad[k] = 0.0;
  const float m = p.beta1 * p.m[k] + (1.0f - p.beta1) * g;
  const float v = p.beta2 * p.v[k] + (1.0f - p.beta2) * g * g;
  p.m[k] = m;
  p.v[k] = v;
  const float mh = m / p.bc1, vh = v / p.bc2;
  p.master[k] -= p.lr * mh / (sqrtf(vh) + p.eps);
}

extern "C" __global__ void __launch_bounds__(256)
hmd_nn_record(const NnRecordParams p) {
  const uint32_t a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= p.n) return;
  reinterpret_cast<float4*>(p.frame_posq)[a] = reinterpret_cast<const float4*>(p.posq)[a];
#pragma unroll
  for (uint32_t d = 0; d < 3; ++d)
    p.frame_target[d * p.n + a] = p.fine_f[d * p.n + a] - p.coarse_f[d * p.n + a];
}

extern "C" __global__ void __launch_bounds__(256)
hmd_nn_diff(const NnDiffParams p) {
  __shared__ double s[2][256];
  const uint32_t chunk = (p.n + gridDim.x - 1) / gridDim.x;
  const uint32_t beg = blockIdx.x * chunk, end = min(beg + chunk, p.n);
  double e = 0.0, b2 = 0.0;
  for (uint32_t i = beg + threadIdx.x; i < end; i += blockDim.x) {
#pragma unroll
    for (uint32_t d = 0; d < 3; ++d) {
      const double a = p.a[d * p.n + i], b = p.b[d * p.n + i];
      e += (a - b) * (a - b);
      b2 += b * b;
    }
  }
  s[0][threadIdx.x] = e;
  s[1][threadIdx.x] = b2;
  __syncthreads();
  for (uint32_t st = blockDim.x / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) {
      s[0][threadIdx.x] += s[0][threadIdx.x + st];
      s[1][threadIdx.x] += s[1][threadIdx.x + st];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    p.partials[blockIdx.x] = s[0][0];
    p.partials[gridDim.x + blockIdx.x] = s[1][0];
  }
}
