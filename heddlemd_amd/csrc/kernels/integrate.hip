// Integrator, constraint and reduction kernels for gfx950.
//
// Reference behaviour: kernels/integrate.cu (velocity Verlet, f32 and the
// compensated (f32 hi, f64 lo) "lossless" variants, :24-314),
// kernels/settle.cu (SETTLE, :47-510), kernels/langevin.cu + philox.cuh
// (BAOAB A and O steps, :13-80; Philox-4x32-10, :25-150) and the KE / virial
// reductions of kernels/nose_hoover.cu:22-104 and kernels/barostat.cu:11-85,
// which here accumulate in FP64 with a fixed reduction tree.
#include "hmd_device.h"

// -------------------------------------------------------- velocity Verlet --
// The arithmetic is that of integrate.cu:24-170 as compiled with FMA
// contraction on: a = F / m (IEEE divide), v + a dt/2 and x + v dt fused
// into one rounding each; the compensated (f32 hi + f64 lo) variant adds the
// f32 product a dt/2 to (hi + lo) in f64 and fuses (v_hi + v_lo) dt into the
// f64 position sum.  Written with explicit fmaf / fma so the rounding does
// not depend on the compiler's contraction choices.

// The state of one atom in registers.  Every sub-step below works on it, so
// that the kernels of one sub-step (load, sub-step, store) and the fused step
// kernels (load once, all sub-steps, store once) run the same operations.
struct HmdAtom {
  float4 pq;
  float v[3];
  double xl[3], vl[3];   // low parts (compensated mode)
  int im[3];             // image counts added by the wraps
};

__device__ inline void hmd_load_pos(const float* posq, const double* lo, uint32_t n, uint32_t i,
                                    HmdAtom& s) {
  s.pq = reinterpret_cast<const float4*>(posq)[i];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    s.xl[d] = lo ? lo[(size_t)d * n + i] : 0.0;
    s.im[d] = 0;
  }
}
__device__ inline void hmd_load_vel(const float* v, const double* lo, uint32_t n, uint32_t i,
                                    HmdAtom& s) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    s.v[d] = v[(size_t)d * n + i];
    s.vl[d] = lo ? lo[(size_t)d * n + i] : 0.0;
  }
}
__device__ inline void hmd_store_pos(float* posq, double* lo, uint32_t n, uint32_t i,
                                     const HmdAtom& s) {
  reinterpret_cast<float4*>(posq)[i] = s.pq;
  if (lo) {
#pragma unroll
    for (int d = 0; d < 3; ++d) lo[(size_t)d * n + i] = s.xl[d];
  }
}
__device__ inline void hmd_store_vel(float* v, double* lo, uint32_t n, uint32_t i,
                                     const HmdAtom& s) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    v[(size_t)d * n + i] = s.v[d];
    if (lo) lo[(size_t)d * n + i] = s.vl[d];
  }
}
__device__ inline void hmd_add_images(int32_t* images, uint32_t n, uint32_t i, const HmdAtom& s) {
#pragma unroll
  for (int d = 0; d < 3; ++d) images[(size_t)d * n + i] += s.im[d];
}

// v += F/m dt/2 (integrate.cu:172-215).
__device__ inline void hmd_vv_kick_state(const VvParams& p, const float f[3], const float m,
                                         HmdAtom& s) {
#pragma clang fp contract(off)
  const float half_dt = p.dt * 0.5f;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const float a = f[d] / m;
    if (p.compensated) {
      const double ext_v = ((double)s.v[d] + s.vl[d]) + (double)(a * half_dt);
      s.v[d] = (float)ext_v;
      s.vl[d] = ext_v - (double)s.v[d];
    } else {
      s.v[d] = fmaf(a, half_dt, s.v[d]);
    }
  }
}

// Wrap into the primary image, counting the images.
__device__ inline void hmd_wrap_state(const HmdLattice& L, HmdAtom& s) {
  int ka, kb, kc;
  hmd_wrap(s.pq.x, s.pq.y, s.pq.z, ka, kb, kc, L);
  s.im[0] += ka;
  s.im[1] += kb;
  s.im[2] += kc;
}

// x += v dt; wrap (integrate.cu:24-170).
__device__ inline void hmd_vv_drift_state(const VvParams& p, HmdAtom& s) {
#pragma clang fp contract(off)
  float x[3] = {s.pq.x, s.pq.y, s.pq.z};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (p.compensated) {
      const double ext_x =
          fma((double)s.v[d] + s.vl[d], (double)p.dt, (double)x[d] + s.xl[d]);
      x[d] = (float)ext_x;
      s.xl[d] = ext_x - (double)x[d];
    } else {
      x[d] = fmaf(s.v[d], p.dt, x[d]);
    }
  }
  s.pq.x = x[0];
  s.pq.y = x[1];
  s.pq.z = x[2];
  hmd_wrap_state(p.L, s);
}

__device__ inline void hmd_load_force(const VvParams& p, uint32_t i, float f[3], float& m) {
#pragma unroll
  for (int d = 0; d < 3; ++d) f[d] = p.f[(size_t)d * p.n + i];
  m = p.m[i];
}

// One atom of the velocity-Verlet plan as its own kernel.
__device__ inline void hmd_vv_kick_drift_atom(const VvParams& p, const uint32_t i) {
  HmdAtom s;
  float f[3], m;
  double* xl = p.compensated ? p.pos_lo : nullptr;
  double* vl = p.compensated ? p.vel_lo : nullptr;
  hmd_load_pos(p.posq, xl, p.n, i, s);
  hmd_load_vel(p.v, vl, p.n, i, s);
  hmd_load_force(p, i, f, m);
  hmd_vv_kick_state(p, f, m, s);
  hmd_vv_drift_state(p, s);
  hmd_store_vel(p.v, vl, p.n, i, s);
  hmd_store_pos(p.posq, xl, p.n, i, s);
  hmd_add_images(p.images, p.n, i, s);
}
__device__ inline void hmd_vv_kick_atom(const VvParams& p, const uint32_t i) {
  HmdAtom s;
  float f[3], m;
  double* vl = p.compensated ? p.vel_lo : nullptr;
  hmd_load_vel(p.v, vl, p.n, i, s);
  hmd_load_force(p, i, f, m);
  hmd_vv_kick_state(p, f, m, s);
  hmd_store_vel(p.v, vl, p.n, i, s);
}

// ------------------------------------------------------------------ SETTLE --
// Every f32 operation rounds once (no contraction), so that the result does
// not depend on how the compiler fuses multiplies and adds in the context a
// group function is inlined into (one kernel per sub-step or the fused step
// kernels).
__device__ inline float hmd_csqrt(float x) { return sqrtf(x > 0.0f ? x : 0.0f); }

// Snapshot of the pre-drift positions (settle.cu:47-67).
__device__ inline void hmd_settle_snapshot_group(const SettleParams& p, const uint32_t g) {
  const float4* ps = reinterpret_cast<const float4*>(p.posq);
  float4* sn = reinterpret_cast<float4*>(p.snapshot);
#pragma unroll
  for (int a = 0; a < 3; ++a) sn[3 * g + a] = ps[p.group_atoms[3 * g + a]];
}

// Apply a position correction to an atom: f32 path or, in compensated mode,
// to the extended (hi + lo) value, re-split.
__device__ inline void hmd_apply_pos(const SettleParams& p, HmdAtom& s, const float cur[3],
                                     const float corr[3], float inv_dt) {
#pragma clang fp contract(off)
  float out[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (p.pos_lo) {
      const double ext = (double)cur[d] + s.xl[d] + (double)corr[d];
      out[d] = (float)ext;
      s.xl[d] = ext - (double)out[d];
      const double ev = (double)s.v[d] + s.vl[d] + (double)(corr[d] * inv_dt);
      s.v[d] = (float)ev;
      s.vl[d] = ev - (double)s.v[d];
    } else {
      out[d] = cur[d] + corr[d];
      s.v[d] = s.v[d] + corr[d] * inv_dt;
    }
  }
  s.pq.x = out[0];
  s.pq.y = out[1];
  s.pq.z = out[2];
}

// Analytic rigid-water position reset (Miyamoto & Kollman, J. Comput.
// Chem. 13(8), 952-962, 1992) with the half-step velocity fix and the
// position-level constraint virial, as settle.cu:145-335.  s: the group's
// atoms, sn: their positions before the drift, cv: the virial.
__device__ inline void hmd_settle_positions_state(const SettleParams& p, HmdAtom s[3],
                                                  const float4 sn[3], const float dt,
                                                  float cv[3]) {
#pragma clang fp contract(off)
  const HmdLattice L = p.L;
  float cur[3][3] = {{s[0].pq.x, s[0].pq.y, s[0].pq.z},
                     {s[1].pq.x, s[1].pq.y, s[1].pq.z},
                     {s[2].pq.x, s[2].pq.y, s[2].pq.z}};
  float snp[3][3] = {{sn[0].x, sn[0].y, sn[0].z},
                     {sn[1].x, sn[1].y, sn[1].z},
                     {sn[2].x, sn[2].y, sn[2].z}};
  // Reference bond vectors and per-atom drifts, minimum-imaged.
  float b0[3] = {snp[1][0] - snp[0][0], snp[1][1] - snp[0][1], snp[1][2] - snp[0][2]};
  float c0[3] = {snp[2][0] - snp[0][0], snp[2][1] - snp[0][1], snp[2][2] - snp[0][2]};
  hmd_min_image(b0[0], b0[1], b0[2], L);
  hmd_min_image(c0[0], c0[1], c0[2], L);
  float xp[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    float dx = cur[a][0] - snp[a][0], dy = cur[a][1] - snp[a][1], dz = cur[a][2] - snp[a][2];
    hmd_min_image(dx, dy, dz, L);
    xp[a][0] = dx; xp[a][1] = dy; xp[a][2] = dz;
  }
  const float m0 = p.m_o, m1 = p.m_h, m2 = p.m_h;
  const float inv_total = 1.0f / (m0 + m1 + m2);
  const float ra = p.ra, rb = p.rb, rc = p.rc;
  // Unconstrained positions relative to the reference oxygen, and the COM.
  float unc[3][3], com[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    unc[0][d] = xp[0][d];
    unc[1][d] = b0[d] + xp[1][d];
    unc[2][d] = c0[d] + xp[2][d];
    com[d] = (unc[0][d] * m0 + unc[1][d] * m1 + unc[2][d] * m2) * inv_total;
  }
  float a1[3], b1[3], c1[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    a1[d] = unc[0][d] - com[d];
    b1[d] = unc[1][d] - com[d];
    c1[d] = unc[2][d] - com[d];
  }
  // Frame: Z' normal to the reference plane, X' from the displaced O.
  float ez[3] = {b0[1] * c0[2] - b0[2] * c0[1], b0[2] * c0[0] - b0[0] * c0[2],
                 b0[0] * c0[1] - b0[1] * c0[0]};
  float ex[3] = {a1[1] * ez[2] - a1[2] * ez[1], a1[2] * ez[0] - a1[0] * ez[2],
                 a1[0] * ez[1] - a1[1] * ez[0]};
  float ey[3] = {ez[1] * ex[2] - ez[2] * ex[1], ez[2] * ex[0] - ez[0] * ex[2],
                 ez[0] * ex[1] - ez[1] * ex[0]};
  const float lx_ = hmd_csqrt(ex[0] * ex[0] + ex[1] * ex[1] + ex[2] * ex[2]);
  const float ly_ = hmd_csqrt(ey[0] * ey[0] + ey[1] * ey[1] + ey[2] * ey[2]);
  const float lz_ = hmd_csqrt(ez[0] * ez[0] + ez[1] * ez[1] + ez[2] * ez[2]);
  const float iex = lx_ > 0.0f ? 1.0f / lx_ : 0.0f;
  const float iey = ly_ > 0.0f ? 1.0f / ly_ : 0.0f;
  const float iez = lz_ > 0.0f ? 1.0f / lz_ : 0.0f;
#pragma unroll
  for (int d = 0; d < 3; ++d) { ex[d] *= iex; ey[d] *= iey; ez[d] *= iez; }
  auto dot = [](const float* u, const float* w) { return u[0] * w[0] + u[1] * w[1] + u[2] * w[2]; };
  const float b0x = dot(ex, b0), b0y = dot(ey, b0), c0x = dot(ex, c0), c0y = dot(ey, c0);
  const float a1z = dot(ez, a1);
  const float b1x = dot(ex, b1), b1y = dot(ey, b1), b1z = dot(ez, b1);
  const float c1x = dot(ex, c1), c1y = dot(ey, c1), c1z = dot(ez, c1);
  // Canonical triangle tilted by (phi, psi), then in-plane rotation theta.
  const float sinphi = a1z / ra;
  const float cosphi = hmd_csqrt(1.0f - sinphi * sinphi);
  const float sinpsi = (b1z - c1z) / (2.0f * rc * cosphi);
  const float cospsi = hmd_csqrt(1.0f - sinpsi * sinpsi);
  const float a2y = ra * cosphi;
  float b2x = -rc * cospsi;
  const float b2y = -rb * cosphi - rc * sinpsi * sinphi;
  const float c2y = -rb * cosphi + rc * sinpsi * sinphi;
  const float hh = 4.0f * b2x * b2x + (b2y - c2y) * (b2y - c2y) + (b1z - c1z) * (b1z - c1z);
  const float d2sq = 4.0f * rc * rc;
  const float delta = 2.0f * b2x + hmd_csqrt(4.0f * b2x * b2x - hh + d2sq);
  b2x -= 0.5f * delta;
  const float al = b2x * (b0x - c0x) + b0y * b2y + c0y * c2y;
  const float be = b2x * (c0y - b0y) + b0x * b2y + c0x * c2y;
  const float ga = b0x * b1y - b1x * b0y + c0x * c1y - c1x * c0y;
  const float ab2 = al * al + be * be;
  const float iab2 = ab2 > 0.0f ? 1.0f / ab2 : 0.0f;
  const float sinth = (al * ga - be * hmd_csqrt(ab2 - ga * ga)) * iab2;
  const float costh = hmd_csqrt(1.0f - sinth * sinth);
  const float pr[3][3] = {{-a2y * sinth, a2y * costh, a1z},
                          {b2x * costh - b2y * sinth, b2x * sinth + b2y * costh, b1z},
                          {-b2x * costh - c2y * sinth, -b2x * sinth + c2y * costh, c1z}};
  const float inv_dt = dt != 0.0f ? 1.0f / dt : 0.0f;
  const float inv_dt2 = inv_dt * inv_dt;
  const float mass[3] = {m0, m1, m2};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    float rcm[3], corr[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      rcm[d] = ex[d] * pr[a][0] + ey[d] * pr[a][1] + ez[d] * pr[a][2];
      corr[d] = (com[d] + rcm[d]) - unc[a][d];
    }
    hmd_apply_pos(p, s[a], cur[a], corr, inv_dt);
    cv[a] = mass[a] * inv_dt2 * (corr[0] * rcm[0] + corr[1] * rcm[1] + corr[2] * rcm[2]);
  }
}

// The same as its own kernel.
__device__ inline void hmd_settle_positions_group(const SettleParams& p, const uint32_t g,
                                                  const float dt) {
  const float4* sm = reinterpret_cast<const float4*>(p.snapshot);
  HmdAtom s[3];
  float4 sn[3];
  float cv[3];
  uint32_t idx[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    idx[a] = p.group_atoms[3 * g + a];
    hmd_load_pos(p.posq, p.pos_lo, p.n, idx[a], s[a]);
    hmd_load_vel(p.v, p.vel_lo, p.n, idx[a], s[a]);
    sn[a] = sm[3 * g + a];
  }
  hmd_settle_positions_state(p, s, sn, dt, cv);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    hmd_store_pos(p.posq, p.pos_lo, p.n, idx[a], s[a]);
    hmd_store_vel(p.v, p.vel_lo, p.n, idx[a], s[a]);
    if (p.constraint_virial) p.constraint_virial[3 * g + a] = cv[a];
  }
}

// Analytic velocity projection: 3x3 Cramer solve for the bond impulses
// (settle.cu:376-490).  The velocity-level constraint virial is added to cv.
__device__ inline void hmd_settle_velocities_state(const SettleParams& p, HmdAtom s[3],
                                                   const float dt, float cv[3]) {
#pragma clang fp contract(off)
  const HmdLattice L = p.L;
  float px[3], py[3], pz[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    px[a] = s[a].pq.x; py[a] = s[a].pq.y; pz[a] = s[a].pq.z;
  }
#pragma unroll
  for (int a = 1; a < 3; ++a) {
    float dx = px[a] - px[0], dy = py[a] - py[0], dz = pz[a] - pz[0];
    hmd_min_image(dx, dy, dz, L);
    px[a] = px[0] + dx; py[a] = py[0] + dy; pz[a] = pz[0] + dz;
  }
  const float io = 1.0f / p.m_o, ih = 1.0f / p.m_h;
  float v[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int d = 0; d < 3; ++d) v[a][d] = s[a].v[d];
  const float r1[3] = {px[0] - px[1], py[0] - py[1], pz[0] - pz[1]};
  const float r2[3] = {px[0] - px[2], py[0] - py[2], pz[0] - pz[2]};
  const float r3[3] = {px[1] - px[2], py[1] - py[2], pz[1] - pz[2]};
  auto dot = [](const float* u, const float* w) { return u[0] * w[0] + u[1] * w[1] + u[2] * w[2]; };
  const float d11 = dot(r1, r1), d22 = dot(r2, r2), d33 = dot(r3, r3);
  const float d12 = dot(r1, r2), d13 = dot(r1, r3), d23 = dot(r2, r3);
  float v01[3], v02[3], v12[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    v01[d] = v[0][d] - v[1][d];
    v02[d] = v[0][d] - v[2][d];
    v12[d] = v[1][d] - v[2][d];
  }
  const float rhs[3] = {-dot(v01, r1), -dot(v02, r2), -dot(v12, r3)};
  const float M[3][3] = {{d11 * (io + ih), d12 * io, -d13 * ih},
                         {d12 * io, d22 * (io + ih), d23 * ih},
                         {-d13 * ih, d23 * ih, 2.0f * d33 * ih}};
  auto det3 = [](const float A[3][3]) {
    return A[0][0] * (A[1][1] * A[2][2] - A[1][2] * A[2][1]) -
           A[0][1] * (A[1][0] * A[2][2] - A[1][2] * A[2][0]) +
           A[0][2] * (A[1][0] * A[2][1] - A[1][1] * A[2][0]);
  };
  const float det = det3(M);
  if (det == 0.0f) return;
  const float idet = 1.0f / det;
  float gg[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float A[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) A[i][j] = (j == c) ? rhs[i] : M[i][j];
    gg[c] = det3(A) * idet;
  }
  float dv[3][3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    dv[0][d] = (gg[0] * r1[d] + gg[1] * r2[d]) * io;
    dv[1][d] = (-gg[0] * r1[d] + gg[2] * r3[d]) * ih;
    dv[2][d] = (-gg[1] * r2[d] - gg[2] * r3[d]) * ih;
  }
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (p.vel_lo) {
        const double ev = (double)v[a][d] + s[a].vl[d] + (double)dv[a][d];
        s[a].v[d] = (float)ev;
        s[a].vl[d] = ev - (double)s[a].v[d];
      } else {
        s[a].v[d] = v[a][d] + dv[a][d];
      }
    }
  if (p.constraint_virial && dt > 0.0f) {
    const float inv_dt = 1.0f / dt;
    const float tm = p.m_o + 2.0f * p.m_h;
    const float cx = (p.m_o * px[0] + p.m_h * px[1] + p.m_h * px[2]) / tm;
    const float cy = (p.m_o * py[0] + p.m_h * py[1] + p.m_h * py[2]) / tm;
    const float cz = (p.m_o * pz[0] + p.m_h * pz[1] + p.m_h * pz[2]) / tm;
    const float mass[3] = {p.m_o, p.m_h, p.m_h};
#pragma unroll
    for (int a = 0; a < 3; ++a)
      cv[a] += mass[a] * inv_dt * (dv[a][0] * (px[a] - cx) + dv[a][1] * (py[a] - cy) +
                                  dv[a][2] * (pz[a] - cz));
  }
}

// The same as its own kernel.
__device__ inline void hmd_settle_velocities_group(const SettleParams& p, const uint32_t g,
                                                   const float dt) {
  HmdAtom s[3];
  float cv[3] = {0.0f, 0.0f, 0.0f};
  uint32_t idx[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    idx[a] = p.group_atoms[3 * g + a];
    hmd_load_pos(p.posq, nullptr, p.n, idx[a], s[a]);
    hmd_load_vel(p.v, p.vel_lo, p.n, idx[a], s[a]);
    if (p.constraint_virial) cv[a] = p.constraint_virial[3 * g + a];
  }
  hmd_settle_velocities_state(p, s, dt, cv);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    hmd_store_vel(p.v, p.vel_lo, p.n, idx[a], s[a]);
    if (p.constraint_virial) p.constraint_virial[3 * g + a] = cv[a];
  }
}

// The group's constraint virial (position level from the last reset plus
// velocity level from the last projection) added to its atoms' virials:
// settle_virial_scatter (kernels/settle.cu:498-510).  Groups are disjoint,
// so the adds need no atomics.
__device__ inline void hmd_settle_virial_group(const SettleParams& p, const uint32_t g) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const uint32_t i = p.group_atoms[3 * g + a];
    p.particle_virial[i] = p.particle_virial[i] + p.constraint_virial[3 * g + a];
  }
}

// --------------------------------------------------------------- Langevin --
// Philox-4x32-10 (Salmon et al., SC'11), as kernels/philox.cuh:25-70.
__device__ inline void hmd_philox(uint32_t k0, uint32_t k1, uint32_t c[4]) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint32_t hi0 = __umulhi(c[0], 0xD2511F53u), lo0 = c[0] * 0xD2511F53u;
    const uint32_t hi2 = __umulhi(c[2], 0xCD9E8D57u), lo2 = c[2] * 0xCD9E8D57u;
    const uint32_t n0 = hi2 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
    c[0] = n0; c[1] = lo2; c[2] = n2; c[3] = lo0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

// Box-Muller cos branch on the first two words with (x + 1/2) 2^-32
// uniforms, f64 internals (philox.cuh:136-150).
__device__ inline double hmd_philox_gaussian_f64(uint32_t sl, uint32_t sh, uint32_t cl,
                                                 uint32_t ch, uint32_t pid, uint32_t axis) {
  uint32_t c[4] = {cl, ch, pid, axis};
  hmd_philox(sl, sh, c);
  const double u1 = ((double)c[0] + 0.5) * (1.0 / 4294967296.0);
  const double u2 = ((double)c[1] + 0.5) * (1.0 / 4294967296.0);
  return sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
}

__device__ inline float hmd_philox_gaussian(uint32_t sl, uint32_t sh, uint32_t cl,
                                            uint32_t ch, uint32_t pid, uint32_t axis) {
  return (float)hmd_philox_gaussian_f64(sl, sh, cl, ch, pid, axis);
}

// A step: x += v dt/2 (one rounding, as the reference's contracted
// x + v * half_dt), wrap (langevin.cu:13-50).
__device__ inline void hmd_lan_drift_half_state(const LangevinParams& p, HmdAtom& s) {
#pragma clang fp contract(off)
  const float h = p.dt * 0.5f;
  s.pq.x = fmaf(s.v[0], h, s.pq.x);
  s.pq.y = fmaf(s.v[1], h, s.pq.y);
  s.pq.z = fmaf(s.v[2], h, s.pq.z);
  hmd_wrap_state(p.L, s);
}

// The normal of atom i's axis d in this step's O sub-step: Philox keyed by
// the seed with counter (draw_lo, draw_hi, particle id, axis).
__device__ inline float hmd_lan_xi(const LangevinParams& p, const unsigned long long step,
                                   const uint32_t i, const uint32_t d) {
  return hmd_philox_gaussian(p.seed_lo, p.seed_hi, (uint32_t)(step & 0xFFFFFFFFull),
                             (uint32_t)(step >> 32), i, d);
}

// O step: v = a v + sigma xi with sigma = sqrt((1 - a^2) kT / m) in f32
// (1 - a^2 and a v + (sigma xi) each rounded once, as the reference's
// contracted expressions) (langevin.cu:52-80).
__device__ inline void hmd_lan_ou_state(const LangevinParams& p, const float m,
                                        const float xi[3], HmdAtom& s) {
#pragma clang fp contract(off)
  const float sig = sqrtf(fmaf(-p.a, p.a, 1.0f) * p.kt / m);
#pragma unroll
  for (int d = 0; d < 3; ++d) s.v[d] = fmaf(p.a, s.v[d], sig * xi[d]);
}

// One atom of the Langevin plan's sub-steps as their own kernels.
__device__ inline void hmd_lan_drift_half_atom(const LangevinParams& p, const uint32_t i) {
  HmdAtom s;
  hmd_load_pos(p.posq, nullptr, p.n, i, s);
  hmd_load_vel(p.v, nullptr, p.n, i, s);
  hmd_lan_drift_half_state(p, s);
  hmd_store_pos(p.posq, nullptr, p.n, i, s);
  hmd_add_images(p.images, p.n, i, s);
}
__device__ inline void hmd_lan_ou_atom(const LangevinParams& p, const uint32_t i) {
  HmdAtom s;
  hmd_load_vel(p.v, nullptr, p.n, i, s);
  const unsigned long long step = *p.step;
  float xi[3];
#pragma unroll 1
  for (uint32_t d = 0; d < 3; ++d) xi[d] = hmd_lan_xi(p, step, i, d);
  hmd_lan_ou_state(p, p.m[i], xi, s);
  hmd_store_vel(p.v, nullptr, p.n, i, s);
}

// ---------------------------------------------------- one kernel per op --
// The reference's sub-steps one launch each (the standalone operator entry
// points and the unfused integrator plan).
__device__ __forceinline__ void hmd_vv_kick_drift_body(const VvParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t i = hmd_bx * blockDim.x + threadIdx.x;
  if (i < p.n) hmd_vv_kick_drift_atom(p, i);
}
HMD_KERNEL(hmd_vv_kick_drift, VvParams, 256)
__device__ __forceinline__ void hmd_vv_kick_body(const VvParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t i = hmd_bx * blockDim.x + threadIdx.x;
  if (i < p.n) hmd_vv_kick_atom(p, i);
}
HMD_KERNEL(hmd_vv_kick, VvParams, 256)
__device__ __forceinline__ void hmd_settle_snapshot_body(const SettleParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t g = hmd_bx * blockDim.x + threadIdx.x;
  if (g < p.n_groups) hmd_settle_snapshot_group(p, g);
}
HMD_KERNEL(hmd_settle_snapshot, SettleParams, 256)
__device__ __forceinline__ void hmd_settle_positions_body(const SettleParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t g = hmd_bx * blockDim.x + threadIdx.x;
  if (g < p.n_groups) hmd_settle_positions_group(p, g, p.dt);
}
HMD_KERNEL(hmd_settle_positions, SettleParams, 256)
__device__ __forceinline__ void hmd_settle_velocities_body(const SettleParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t g = hmd_bx * blockDim.x + threadIdx.x;
  if (g < p.n_groups) hmd_settle_velocities_group(p, g, p.dt);
}
HMD_KERNEL(hmd_settle_velocities, SettleParams, 256)
__device__ __forceinline__ void hmd_settle_virial_body(const SettleParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t g = hmd_bx * blockDim.x + threadIdx.x;
  if (g < p.n_groups) hmd_settle_virial_group(p, g);
}
HMD_KERNEL(hmd_settle_virial, SettleParams, 256)
__device__ __forceinline__ void hmd_lan_drift_half_body(const LangevinParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t i = hmd_bx * blockDim.x + threadIdx.x;
  if (i < p.n) hmd_lan_drift_half_atom(p, i);
}
HMD_KERNEL(hmd_lan_drift_half, LangevinParams, 256)
__device__ __forceinline__ void hmd_lan_ou_body(const LangevinParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t i = hmd_bx * blockDim.x + threadIdx.x;
  if (i < p.n) hmd_lan_ou_atom(p, i);
}
HMD_KERNEL(hmd_lan_ou, LangevinParams, 256)

// ------------------------------------------------------ fused step kernels --
// The integrator's sub-steps between two force evaluations in one launch.
// One thread owns a SETTLE group and runs every sub-step for its three atoms
// in plan order (the constraint couples only the atoms of one group, so no
// other thread's data is read); free atoms (free_atoms[k], atom k when null)
// have a thread each.  Each atom sees the same operations, in the same order
// and with the same rounding, as in the one-kernel-per-sub-step plan.
//
// Bound by latency: a box of 65,536 groups is one wave a SIMD.  The state is
// loaded once, kept in registers through the sub-steps and stored once (the
// sub-steps' own loads and stores made a chain of ten memory round trips in
// the Langevin kernel), and the groups are spread over workgroups of one
// wave.  Traced at 65,536 groups: first velocity-Verlet kernel 21.8 -> 13.8
// us (compensated, 41 MB), last kick 11.2 -> 7.9 us; Langevin kernel 28.9 ->
// 14.0 us at 8,192 groups, 25.5 -> 13.6 us at 216.
__device__ inline bool hmd_unit(const StepParams& p, uint32_t u, uint32_t& g, uint32_t& atom) {
  if (u < p.st.n_groups) { g = u; return true; }
  const uint32_t k = u - p.st.n_groups;
  g = HMD_SENTINEL;
  atom = k;
  if (k >= p.n_free) return false;
  if (p.free_atoms) atom = p.free_atoms[k];
  return true;
}

// The neighbour list's skin check (hmd_nbl_displacement, the same f32
// arithmetic) on an atom's final position of the step, folded into the
// kernel that wrote it: one dependent launch less before the force
// evaluation.  r: the atom's position at the last list build.
__device__ inline bool hmd_step_displaced(const NblDispParams& d, const float4 a, const float4 r) {
#pragma clang fp contract(off)
  float dx = a.x - r.x, dy = a.y - r.y, dz = a.z - r.z;
  hmd_min_image(dx, dy, dz, d.L);
  const float d2 = dx * dx + dy * dy + dz * dz;
  return d2 > d.threshold_sq;
}
__device__ inline float4 hmd_step_ref(const NblDispParams& d, uint32_t atom) {
  return d.status ? reinterpret_cast<const float4*>(d.ref_pos)[atom]
                  : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// A group's atoms loaded at once.
struct HmdGroup {
  HmdAtom s[3];
  uint32_t idx[3];
  float f[3][3], m[3];
};
__device__ inline void hmd_load_group(const StepParams& p, const uint32_t g, bool pos_lo,
                                      HmdGroup& G) {
  double* xl = p.vv.compensated && pos_lo ? p.vv.pos_lo : nullptr;
  double* vl = p.vv.compensated ? p.vv.vel_lo : nullptr;
#pragma unroll
  for (int a = 0; a < 3; ++a) G.idx[a] = p.st.group_atoms[3 * g + a];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    hmd_load_pos(p.vv.posq, xl, p.vv.n, G.idx[a], G.s[a]);
    hmd_load_vel(p.vv.v, vl, p.vv.n, G.idx[a], G.s[a]);
    hmd_load_force(p.vv, G.idx[a], G.f[a], G.m[a]);
  }
}
// Positions, velocities and images back, with the skin check.
__device__ inline void hmd_store_group(const StepParams& p, const HmdGroup& G,
                                       const float4 ref[3]) {
  double* xl = p.vv.compensated ? p.vv.pos_lo : nullptr;
  double* vl = p.vv.compensated ? p.vv.vel_lo : nullptr;
  bool moved = false;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    hmd_store_pos(p.vv.posq, xl, p.vv.n, G.idx[a], G.s[a]);
    hmd_store_vel(p.vv.v, vl, p.vv.n, G.idx[a], G.s[a]);
    hmd_add_images(p.vv.images, p.vv.n, G.idx[a], G.s[a]);
    moved |= hmd_step_displaced(p.disp, G.s[a].pq, ref[a]);
  }
  if (moved && p.disp.status) atomicOr(p.disp.status, HMD_STATUS_DISPLACED);
}
__device__ inline void hmd_snap(const HmdGroup& G, float4 sn[3]) {
#pragma unroll
  for (int a = 0; a < 3; ++a) sn[a] = G.s[a].pq;
}

// velocity Verlet: [snapshot] kick-drift [SETTLE positions] [skin check]
__device__ __forceinline__ void hmd_step_vv_first_body(const StepParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t u = hmd_bx * blockDim.x + threadIdx.x;
  uint32_t g, atom;
  if (!hmd_unit(p, u, g, atom)) return;
  if (g != HMD_SENTINEL) {
    HmdGroup G;
    float4 ref[3], sn[3];
    float cv[3];
    hmd_load_group(p, g, true, G);
#pragma unroll
    for (int a = 0; a < 3; ++a) ref[a] = hmd_step_ref(p.disp, G.idx[a]);
    hmd_snap(G, sn);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      hmd_vv_kick_state(p.vv, G.f[a], G.m[a], G.s[a]);
      hmd_vv_drift_state(p.vv, G.s[a]);
    }
    hmd_settle_positions_state(p.st, G.s, sn, p.dt, cv);
    hmd_store_group(p, G, ref);
    if (p.st.particle_virial) {   // read by the step's last kernel only then
#pragma unroll
      for (int a = 0; a < 3; ++a) p.st.constraint_virial[3 * g + a] = cv[a];
    }
  } else {
    hmd_vv_kick_drift_atom(p.vv, atom);
    if (p.disp.status &&
        hmd_step_displaced(p.disp, reinterpret_cast<const float4*>(p.vv.posq)[atom],
                           hmd_step_ref(p.disp, atom)))
      atomicOr(p.disp.status, HMD_STATUS_DISPLACED);
  }
}
HMD_KERNEL(hmd_step_vv_first, StepParams, 256)

// Langevin BAOAB up to the force evaluation: B [SETTLE v] [snapshot] A
// [SETTLE x, dt/2] O [SETTLE v] [snapshot] A [SETTLE x, dt/2] [skin check].
// A workgroup of 256 threads takes HMD_BAOA_GROUPS groups: all its threads
// draw the groups' normals first (nine a group; a Philox block and an FP64
// log, square root and cosine each, half of the kernel's time when the
// group's own thread drew them one after the other), then a thread a group
// runs the sub-steps: one full wave (16 groups a workgroup, which draw in one
// round, took 1.1 us a step more at 216 and at 1,000 groups, 1.6 at 4,096, 7 at
// 16,384).  Blocks past group_blocks take 256 free atoms each.
__device__ __forceinline__ void hmd_step_baoa_body(const StepParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  __shared__ float s_xi[9 * HMD_BAOA_GROUPS];
  const unsigned long long step = *p.lan.step;
  if (hmd_bx >= p.group_blocks) {
    const uint32_t k = (hmd_bx - p.group_blocks) * blockDim.x + threadIdx.x;
    if (k >= p.n_free) return;
    const uint32_t i = p.free_atoms ? p.free_atoms[k] : k;
    HmdAtom s;
    float f[3], m, xi[3];
    hmd_load_pos(p.lan.posq, nullptr, p.lan.n, i, s);
    hmd_load_vel(p.lan.v, nullptr, p.lan.n, i, s);
    hmd_load_force(p.vv, i, f, m);
    const float4 ref = hmd_step_ref(p.disp, i);
#pragma unroll 1
    for (uint32_t d = 0; d < 3; ++d) xi[d] = hmd_lan_xi(p.lan, step, i, d);
    hmd_vv_kick_state(p.vv, f, m, s);
    hmd_lan_drift_half_state(p.lan, s);
    hmd_lan_ou_state(p.lan, m, xi, s);
    hmd_lan_drift_half_state(p.lan, s);
    hmd_store_pos(p.lan.posq, nullptr, p.lan.n, i, s);
    hmd_store_vel(p.lan.v, nullptr, p.lan.n, i, s);
    hmd_add_images(p.lan.images, p.lan.n, i, s);
    if (p.disp.status && hmd_step_displaced(p.disp, s.pq, ref))
      atomicOr(p.disp.status, HMD_STATUS_DISPLACED);
    return;
  }
  const uint32_t g0 = hmd_bx * HMD_BAOA_GROUPS;
  const uint32_t ng = min(HMD_BAOA_GROUPS, p.st.n_groups - g0);
  const bool mine = threadIdx.x < ng;
  const uint32_t g = g0 + threadIdx.x;
  HmdGroup G;
  float4 ref[3], sn[3];
  if (mine) {
    hmd_load_group(p, g, false, G);
#pragma unroll
    for (int a = 0; a < 3; ++a) ref[a] = hmd_step_ref(p.disp, G.idx[a]);
  }
  for (uint32_t k = threadIdx.x; k < 9u * ng; k += blockDim.x) {
    const uint32_t a = k / 3u, d = k - 3u * a;   // a: atom of the block's groups
    s_xi[k] = hmd_lan_xi(p.lan, step, p.st.group_atoms[3u * g0 + a], d);
  }
  __syncthreads();
  if (!mine) return;
  const float h = 0.5f * p.dt;
  float cv[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int a = 0; a < 3; ++a) hmd_vv_kick_state(p.vv, G.f[a], G.m[a], G.s[a]);
  hmd_settle_velocities_state(p.st, G.s, p.dt, cv);
  hmd_snap(G, sn);
#pragma unroll
  for (int a = 0; a < 3; ++a) hmd_lan_drift_half_state(p.lan, G.s[a]);
  hmd_settle_positions_state(p.st, G.s, sn, h, cv);
#pragma unroll
  for (int a = 0; a < 3; ++a)
    hmd_lan_ou_state(p.lan, G.m[a], &s_xi[9u * threadIdx.x + 3u * a], G.s[a]);
  hmd_settle_velocities_state(p.st, G.s, p.dt, cv);
  hmd_snap(G, sn);
#pragma unroll
  for (int a = 0; a < 3; ++a) hmd_lan_drift_half_state(p.lan, G.s[a]);
  hmd_settle_positions_state(p.st, G.s, sn, h, cv);
  hmd_store_group(p, G, ref);
  if (p.st.particle_virial) {   // read by the step's last kernel only then
#pragma unroll
    for (int a = 0; a < 3; ++a) p.st.constraint_virial[3 * g + a] = cv[a];
  }
}
HMD_KERNEL(hmd_step_baoa, StepParams, 256)

// after the force evaluation: kick [SETTLE velocities]; the Langevin draw
// counter (read by this step's O sub-step) advances here
__device__ __forceinline__ void hmd_step_kick_last_body(const StepParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t u = hmd_bx * blockDim.x + threadIdx.x;
  if (u == 0 && p.counter) p.counter[0] += 1ull;
  uint32_t g, atom;
  if (!hmd_unit(p, u, g, atom)) return;
  if (g != HMD_SENTINEL) {
    HmdGroup G;
    float cv[3] = {0.0f, 0.0f, 0.0f}, w[3] = {0.0f, 0.0f, 0.0f};
    hmd_load_group(p, g, false, G);
    if (p.st.particle_virial) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        cv[a] = p.st.constraint_virial[3 * g + a];
        w[a] = p.st.particle_virial[G.idx[a]];
      }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) hmd_vv_kick_state(p.vv, G.f[a], G.m[a], G.s[a]);
    hmd_settle_velocities_state(p.st, G.s, p.dt, cv);
    double* vl = p.vv.compensated ? p.vv.vel_lo : nullptr;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      hmd_store_vel(p.vv.v, vl, p.vv.n, G.idx[a], G.s[a]);
      if (p.st.particle_virial) p.st.particle_virial[G.idx[a]] = w[a] + cv[a];
    }
  } else {
    hmd_vv_kick_atom(p.vv, atom);
  }
}
HMD_KERNEL(hmd_step_kick_last, StepParams, 256)

__device__ __forceinline__ void hmd_counter_increment_body(const CounterParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  if (threadIdx.x == 0 && hmd_bx == 0) p.counter[0] += 1ull;
}
HMD_KERNEL(hmd_counter_increment, CounterParams, 64)

// -------------------------------------------------------------- reductions --
// Fixed-shape FP64 reduction: block b sums a fixed contiguous chunk in a
// fixed per-thread order and a fixed LDS tree; hmd_reduce_final sums the
// block partials the same way.  Mode 0: sum x[0..n); mode 1: kinetic energy
// 0.5 m |v|^2 (nose_hoover.cu:22-104 and barostat.cu:11-85 restated in
// FP64).
__device__ __forceinline__ void hmd_reduce_partial_body(const ReduceParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  __shared__ double s[256];
  const uint32_t chunk = (p.n + hmd_gx - 1) / hmd_gx;
  const uint32_t beg = hmd_bx * chunk, end = min(beg + chunk, p.n);
  double acc = 0.0;
  for (uint32_t i = beg + threadIdx.x; i < end; i += blockDim.x) {
    if (p.mode == 0) {
      acc += (double)p.x[i];
    } else {
      const double vx = p.v[i], vy = p.v[p.n + i], vz = p.v[2 * p.n + i];
      acc += 0.5 * (double)p.m[i] * (vx * vx + vy * vy + vz * vz);
    }
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (uint32_t st = blockDim.x / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) s[threadIdx.x] += s[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) p.partials[hmd_bx] = s[0];
}
HMD_KERNEL(hmd_reduce_partial, ReduceParams, 256)

__device__ __forceinline__ void hmd_reduce_final_body(const ReduceParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  __shared__ double s[256];
  double acc = 0.0;
  for (uint32_t i = threadIdx.x; i < p.n_blocks; i += blockDim.x) acc += p.partials[i];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (uint32_t st = blockDim.x / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) s[threadIdx.x] += s[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) p.out[0] = s[0];
}
HMD_KERNEL(hmd_reduce_final, ReduceParams, 256)

// ------------------------------------------------------------------- CSVR --
// Stochastic velocity rescaling (Bussi, Donadio & Parrinello, J. Chem. Phys.
// 126, 014101 (2007)) as kernels/nose_hoover.cu:181-360 applies it after a
// step: with the kinetic energy K, N_f = g_dof and the normals xi_i of
// Philox (seed, draw counter, i, 0),
//   K' = c K + (kT/2)(1 - c)(sum_{i=1}^{N_f-1} xi_i^2 + xi_0^2)
//        + 2 xi_0 sqrt(c (1 - c) K kT/2),
// v <- sqrt(K'/K) v, and the injected energy K' - K accumulates for the
// conserved quantity.  All on the device (capturable); the draw counter
// advances once per application.  Sums: a fixed chunk per block, a fixed
// lane stride and LDS tree per block, a fixed tree over the blocks.
__device__ inline double hmd_block_sum(double v, double* s) {
  s[threadIdx.x] = v;
  __syncthreads();
  for (uint32_t st = blockDim.x / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) s[threadIdx.x] += s[threadIdx.x + st];
    __syncthreads();
  }
  return s[0];
}

__device__ __forceinline__ void hmd_csvr_sample_body(const CsvrParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  __shared__ double s[256];
  const unsigned long long ctr = *p.counter;
  const uint32_t cl = (uint32_t)(ctr & 0xFFFFFFFFull), ch = (uint32_t)(ctr >> 32);
  const uint32_t m = p.g_dof > 0u ? p.g_dof - 1u : 0u;   // draws i = 1 .. g_dof - 1
  const uint32_t chunk = (m + hmd_gx - 1u) / hmd_gx;
  const uint32_t beg = hmd_bx * chunk, end = min(beg + chunk, m);
  double acc = 0.0;
  for (uint32_t j = beg + threadIdx.x; j < end; j += blockDim.x) {
    const double xi = hmd_philox_gaussian_f64(p.seed_lo, p.seed_hi, cl, ch, j + 1u, 0u);
    acc += xi * xi;
  }
  const double t = hmd_block_sum(acc, s);
  if (threadIdx.x == 0) p.partials[hmd_bx] = t;
}
HMD_KERNEL(hmd_csvr_sample, CsvrParams, 256)

__device__ __forceinline__ void hmd_csvr_finish_body(const CsvrParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  __shared__ double s[256];
  double acc = 0.0;
  for (uint32_t i = threadIdx.x; i < p.n_partials; i += blockDim.x) acc += p.partials[i];
  const double sum = hmd_block_sum(acc, s);
  if (threadIdx.x == 0) {
    const unsigned long long ctr = *p.counter;
    const uint32_t cl = (uint32_t)(ctr & 0xFFFFFFFFull), ch = (uint32_t)(ctr >> 32);
    const double r = hmd_philox_gaussian_f64(p.seed_lo, p.seed_hi, cl, ch, 0u, 0u);
    const double k = *p.ke;
    const double cross = k > 0.0 ? 2.0 * r * sqrt(p.c * p.one_minus_c * k * p.kt_half) : 0.0;
    double kn = p.c * k + p.kt_half * p.one_minus_c * (sum + r * r) + cross;
    if (!isfinite(kn) || kn <= 0.0) kn = k;
    const double f = (k > 0.0 && kn != k) ? sqrt(kn / k) : 1.0;
    p.factor[0] = (float)f;
    p.injection[0] += kn - k;
    *p.counter = ctr + 1ull;
  }
}
HMD_KERNEL(hmd_csvr_finish, CsvrParams, 256)

// v <- factor v (f32, as rescale_velocities_device_factor); in compensated
// mode the extended velocity hi + lo is scaled in f64 and split again.
__device__ __forceinline__ void hmd_csvr_rescale_body(const CsvrParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t i = hmd_bx * blockDim.x + threadIdx.x;
  if (i >= p.n) return;
  const float f = p.factor[0];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const size_t k = (size_t)d * p.n + i;
    if (p.vel_lo) {
      const double ev = ((double)p.v[k] + p.vel_lo[k]) * (double)f;
      const float vh = (float)ev;
      p.vel_lo[k] = ev - (double)vh;
      p.v[k] = vh;
    } else {
      p.v[k] = p.v[k] * f;
    }
  }
}
HMD_KERNEL(hmd_csvr_rescale, CsvrParams, 256)

// ------------------------------------------------------- c-rescale --
// Stochastic cell rescaling (Bernetti & Bussi, J. Chem. Phys. 153, 114107
// (2020)), one isotropic move per step as kernels/barostat.cu:169-227 makes
// it, in FP64 on one thread: with the kinetic energy K, the virial sum W and
// the volume V,
//   P   = (2K + W) / (3V),
//   mu3 = 1 - beta (dt / tau)(P_target - P) + sqrt(2 beta kT dt / (tau V)) r,
// r the Philox normal (seed, draw counter, 0, 0); mu3 is floored at mu3_min
// and mu = cbrt(mu3).  The energy P_target (V mu3 - V) accumulates for the
// conserved quantity and the draw counter advances once.
__device__ __forceinline__ void hmd_crescale_mu_body(const CRescaleParams& p,
    const uint32_t hmd_bx, const uint32_t hmd_gx) {
  if (threadIdx.x != 0 || hmd_bx != 0) return;
  const unsigned long long ctr = *p.counter;
  const uint32_t cl = (uint32_t)(ctr & 0xFFFFFFFFull), ch = (uint32_t)(ctr >> 32);
  const double v = p.v_pre;
  const double pressure = (2.0 * p.ke[0] + p.w[0]) / (3.0 * v);
  const double r = hmd_philox_gaussian_f64(p.seed_lo, p.seed_hi, cl, ch, 0u, 0u);
  const double drift = -p.beta * (p.dt / p.tau) * (p.p_target - pressure);
  const double noise = sqrt(2.0 * p.beta * p.kt * p.dt / (p.tau * v));
  double mu3 = 1.0 + drift + noise * r;
  mu3 = mu3 > p.mu3_min ? mu3 : p.mu3_min;
  const double v_post = v * mu3;
  p.state[0] = cbrt(mu3);
  p.state[1] = pressure;
  p.state[2] = v_post;
  p.state[3] += p.p_target * (v_post - v);
  *p.counter = ctr + 1ull;
}
HMD_KERNEL(hmd_crescale_mu, CRescaleParams, 64)

// x <- (float) mu x for every atom (rescale_positions_device_factor,
// kernels/barostat.cu:93-107); fractional coordinates and image counts are
// unchanged.  In compensated mode the extended position hi + lo is scaled in
// f64 and split again.
__device__ __forceinline__ void hmd_crescale_positions_body(const CRescaleParams& p,
    const uint32_t hmd_bx, const uint32_t hmd_gx) {
  const uint32_t i = hmd_bx * blockDim.x + threadIdx.x;
  if (i >= p.n) return;
  const float f = (float)p.state[0];
  float4 pq = reinterpret_cast<float4*>(p.posq)[i];
  float x[3] = {pq.x, pq.y, pq.z};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (p.pos_lo) {
      const size_t k = (size_t)d * p.n + i;
      const double e = ((double)x[d] + p.pos_lo[k]) * (double)f;
      x[d] = (float)e;
      p.pos_lo[k] = e - (double)x[d];
    } else {
      x[d] = x[d] * f;
    }
  }
  pq.x = x[0]; pq.y = x[1]; pq.z = x[2];
  reinterpret_cast<float4*>(p.posq)[i] = pq;
}
HMD_KERNEL(hmd_crescale_positions, CRescaleParams, 256)

// ------------------------------------------------------- steepest descent --
// x += h F, with |h F| capped at max_step per atom, then wrap (setup-time
// relaxation of synthetic lattices; the reference relaxes its examples with
// its steepest-descent minimizer, src/minimizer/).
__device__ __forceinline__ void hmd_sd_step_body(const SdParams& p, const uint32_t hmd_bx,
    const uint32_t hmd_gx) {
  const uint32_t i = hmd_bx * blockDim.x + threadIdx.x;
  if (i >= p.n) return;
  float4 pq = reinterpret_cast<float4*>(p.posq)[i];
  float d[3] = {p.f[i] * p.h, p.f[p.n + i] * p.h, p.f[2 * p.n + i] * p.h};
  const float len = sqrtf(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
  const float s = len > p.max_step ? p.max_step / len : 1.0f;
  float x = pq.x + d[0] * s, y = pq.y + d[1] * s, z = pq.z + d[2] * s;
  int ka, kb, kc;
  hmd_wrap(x, y, z, ka, kb, kc, p.L);
  pq.x = x; pq.y = y; pq.z = z;
  reinterpret_cast<float4*>(p.posq)[i] = pq;
}
HMD_KERNEL(hmd_sd_step, SdParams, 256)
