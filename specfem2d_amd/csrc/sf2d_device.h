// Device code shared by the element kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "sf2d_mesh.h"

namespace sf2d {

__device__ __forceinline__ void atomic_add_f32(float* p, float v) { unsafeAtomicAdd(p, v); }

constexpr int NXCD = 8;  // gfx950: 8 accelerator complex dies, workgroups dispatched round-robin

// Load through a 32-bit byte offset from a uniform base (global_load with saddr + voffset).  Within its reach are a field
// and an element array of 4 bytes a point, below 4 GiB (checked when the handle is prepared).  The element arrays of 8 and
// 16 bytes a point are longer from 21.5 and 10.7 million elements on: offsets into them count from at_element, the first
// element of a chain, tower or patch, or the kernel is chosen only where they are short (tower_geometry, shot_minor_fits).
template <typename T>
__device__ __forceinline__ T ld_off(const T* base, unsigned byte_off) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + byte_off);
}

// One point's viscoelastic update (3 standard linear solids): the memory variables ev (e1, e11, e13 per solid)
// advance by the recursive convolution of compute_attenuation_viscoelastic.f90:93-121 with the coefficient set
// cf[k] = {A_kappa, B_kappa, A_mu, B_mu}, the previous strains ov (dux_dxl, duz_dzl, dux_dzl + duz_dxl) become
// this step's, and the stress takes the unrelaxed-moduli correction.
__device__ __forceinline__ void attenuate_point(const float4 (&cf)[3], float (&ev)[9], float (&ov)[3], float kap,
                                                float mu, float dux_dxl, float dux_dzl, float duz_dxl, float duz_dzl,
                                                float& sxx, float& sxz, float& szz) {
  const float th = dux_dxl + duz_dzl;
  const float oxx = ov[0], ozz = ov[1], oxz = ov[2];
  const float th_old = oxx + ozz;
  float e1s = 0.f, e11s = 0.f, e13s = 0.f;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float a1 = cf[k].x, b1 = cf[k].y, a2 = cf[k].z, b2 = cf[k].w;
    const float e1 = a1 * a1 * ev[3 * k] + b1 * (th + a1 * th_old);
    const float e11 = a2 * a2 * ev[3 * k + 1] + b2 * (dux_dxl - 0.5f * th + a2 * (oxx - 0.5f * th_old));
    const float e13 = a2 * a2 * ev[3 * k + 2] + b2 * (dux_dzl + duz_dxl + a2 * oxz);
    ev[3 * k] = e1;
    ev[3 * k + 1] = e11;
    ev[3 * k + 2] = e13;
    e1s += e1;
    e11s += e11;
    e13s += e13;
  }
  ov[0] = dux_dxl;
  ov[1] = duz_dzl;
  ov[2] = dux_dzl + duz_dxl;
  sxx += kap * e1s + 2.f * mu * e11s;
  sxz += mu * e13s;
  szz += kap * e1s - 2.f * mu * e11s;
}

// A point's attenuation state as three float4 planes of [3][ne] (ne = element points): the 9 memory variables then
// the 3 previous strains, {e1, e11, e13} of solid 1, 2, 3 and {dux_dxl, duz_dzl, dux_dzl + duz_dxl}
__device__ __forceinline__ void att_load(const float* st, long ne, size_t l, float (&ev)[9], float (&ov)[3]) {
  const float4* s4 = reinterpret_cast<const float4*>(st);
  const float4 a = s4[l], b = s4[(size_t)ne + l], c = s4[2 * (size_t)ne + l];
  ev[0] = a.x; ev[1] = a.y; ev[2] = a.z; ev[3] = a.w;
  ev[4] = b.x; ev[5] = b.y; ev[6] = b.z; ev[7] = b.w;
  ev[8] = c.x; ov[0] = c.y; ov[1] = c.z; ov[2] = c.w;
}
__device__ __forceinline__ void att_store(float* st, long ne, size_t l, const float (&ev)[9], const float (&ov)[3]) {
  float4* s4 = reinterpret_cast<float4*>(st);
  s4[l] = make_float4(ev[0], ev[1], ev[2], ev[3]);
  s4[(size_t)ne + l] = make_float4(ev[4], ev[5], ev[6], ev[7]);
  s4[2 * (size_t)ne + l] = make_float4(ev[8], ov[0], ov[1], ov[2]);
}

// Stacey absorbing faces (elements in device order, i and j 0-based, -1 for a point owned by the neighbouring edge)
struct StaceyFaces {
  int nabs;
  const int *ispec, *ij;
  const float *normal, *jacw;
  const int *ibool, *is_elastic;
  const float *rho_vp, *rho_vs;
};

inline StaceyFaces stacey_faces(const Mesh* mp) {
  return {mp->num_abs, mp->d_abs_ispec, mp->d_abs_ij, mp->d_abs_normal, mp->d_abs_jacw, mp->d_ibool,
          mp->d_ispec_is_elastic, mp->d_rho_vp, mp->d_rho_vs};
}

// Stacey absorbing traction of face point idx (face idx / 5), subtracted from accel and returned
// (src/gpu/kernels/compute_stacey_elastic_kernel.cu:37-150, src/specfem2D/compute_stacey_elastic.f90:34-1001)
__device__ __forceinline__ float2 stacey_traction(const StaceyFaces& F, int idx, const float2* __restrict__ veloc,
                                                  float* __restrict__ accel, int ps) {
  const int f = idx / NGLL;
  if (f >= F.nabs) return make_float2(0.f, 0.f);
  const int i = F.ij[2 * idx], j = F.ij[2 * idx + 1];
  if (i < 0 || j < 0) return make_float2(0.f, 0.f);  // duplicated corner point, handled by the neighbouring edge
  const int ispec = F.ispec[f];
  if (!F.is_elastic[ispec]) return make_float2(0.f, 0.f);
  const size_t l = (size_t)ispec * NGLL2 + j * NGLL + i;
  const long g = (long)F.ibool[l] * ps;
  const float2 v = veloc[g];
  const float nx = F.normal[2 * idx], nz = F.normal[2 * idx + 1];
  const float vn = nx * v.x + nz * v.y;
  const float rvp = F.rho_vp[l], rvs = F.rho_vs[l];
  const float tx = rvp * vn * nx + rvs * (v.x - vn * nx);
  const float tz = rvp * vn * nz + rvs * (v.y - vn * nz);
  const float w = F.jacw[idx];
  const float fx = tx * w, fz = tz * w;
  atomic_add_f32(&accel[2 * (size_t)g], -fx);
  atomic_add_f32(&accel[2 * (size_t)g + 1], -fz);
  return make_float2(fx, fz);
}

// collocated force sources, one time function each ([nstep][nsrc])
struct SourceSet {
  int nsrc;
  const int *ispec, *is_elastic, *ibool;
  const float *arrays, *stf;
};

inline SourceSet source_set(const Mesh* mp) {
  return {mp->nsources_local, mp->d_ispec_selected_source, mp->d_ispec_is_elastic, mp->d_ibool, mp->d_sourcearrays,
          mp->d_stf};
}

// point p of source s at time sample it, added to accel (src/gpu/kernels/compute_add_sources_kernel.cu:37-70)
__device__ __forceinline__ void source_force(const SourceSet& S, int s, int p, int it, float* __restrict__ accel,
                                             int ps) {
  if (p >= NGLL2) return;
  const int ispec = S.ispec[s];
  if (!S.is_elastic[ispec]) return;
  const long g = (long)S.ibool[(size_t)ispec * NGLL2 + p] * ps;
  const float f = S.stf[(size_t)it * S.nsrc + s];
  atomic_add_f32(&accel[2 * (size_t)g], S.arrays[(s * NGLL2 + p) * 2] * f);
  atomic_add_f32(&accel[2 * (size_t)g + 1], S.arrays[(s * NGLL2 + p) * 2 + 1] * f);
}

struct ReceiverSet {
  int nrec, nlength;
  const int *ispec, *ibool;
  const float *xir, *gammar, *cosrot, *sinrot;
};

inline ReceiverSet receiver_set(const Mesh* mp) {
  return {mp->nrec_local, mp->nlength_seismogram, mp->d_ispec_selected_rec, mp->d_ibool, mp->d_xir, mp->d_gammar,
          mp->d_cosrot, mp->d_sinrot};
}

// sample cur of receiver r: Lagrange interpolation over the wave's lanes p, FP64 accumulation, rotation
// (src/gpu/kernels/compute_elastic_seismogram_kernel.cu:69-192; compute_interpolated_dva.f90)
__device__ __forceinline__ void record_receiver(const ReceiverSet& R, int r, int p, int cur,
                                                const float2* __restrict__ field, float* __restrict__ dst, int ps) {
  if (r >= R.nrec) return;
  double vx = 0.0, vz = 0.0;
  if (p < NGLL2) {
    const int i = p % NGLL, j = p / NGLL;
    const long g = (long)R.ibool[(size_t)R.ispec[r] * NGLL2 + p] * ps;
    const double h = (double)(R.xir[i * R.nrec + r] * R.gammar[j * R.nrec + r]);
    const float2 u = field[g];
    vx = (double)u.x * h;
    vz = (double)u.y * h;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    vx += __shfl_xor(vx, off, 64);
    vz += __shfl_xor(vz, off, 64);
  }
  if (p == 0) {
    const double c = R.cosrot[r], s = R.sinrot[r];
    dst[(size_t)r * R.nlength + cur] = (float)(c * vx + s * vz);
    dst[((size_t)R.nrec + r) * R.nlength + cur] = (float)(-s * vx + c * vz);
  }
}

// stored Stacey terms ([face point][2]) of the forward run, subtracted from the reconstructed field's force
// (compute_stacey_viscoelastic.f90, the backward part)
__device__ __forceinline__ void stored_traction(const StaceyFaces& F, int idx, const float2* __restrict__ store,
                                                float* __restrict__ accel) {
  const int f = idx / NGLL;
  if (f >= F.nabs) return;
  const int i = F.ij[2 * idx], j = F.ij[2 * idx + 1];
  if (i < 0 || j < 0) return;
  const int ispec = F.ispec[f];
  if (!F.is_elastic[ispec]) return;
  const size_t g = (size_t)F.ibool[(size_t)ispec * NGLL2 + j * NGLL + i];
  const float2 t = store[idx];
  atomic_add_f32(&accel[2 * g], -t.x);
  atomic_add_f32(&accel[2 * g + 1], -t.y);
}

// adjoint source of receiver r at time sample it (adj: [2][nstep][nrec]), added to accel at its element's point p
// (compute_add_sources_viscoelastic_cuda.cu:131)
__device__ __forceinline__ void adjoint_source(const ReceiverSet& R, const int* __restrict__ is_elastic, int r, int p,
                                               int it, int nstep, const float* __restrict__ adj,
                                               float* __restrict__ accel) {
  if (r >= R.nrec || p >= NGLL2) return;
  const int ispec = R.ispec[r];
  if (!is_elastic[ispec]) return;
  const int i = p % NGLL, j = p / NGLL;
  const size_t g = (size_t)R.ibool[(size_t)ispec * NGLL2 + p];
  const float h = R.xir[i * R.nrec + r] * R.gammar[j * R.nrec + r];
  atomic_add_f32(&accel[2 * g], adj[(size_t)it * R.nrec + r] * h);
  atomic_add_f32(&accel[2 * g + 1], adj[((size_t)nstep + it) * R.nrec + r] * h);
}

// point p of receiver r's residual {x, z} (its rotated components) into D, the adjoint of record_receiver
__device__ __forceinline__ void adjoint_receiver(const ReceiverSet& R, int r, int p, const float* __restrict__ res,
                                                 float* __restrict__ D, int ps) {
  if (r >= R.nrec || p >= NGLL2) return;
  const int i = p % NGLL, j = p / NGLL;
  const float px = res[2 * r], pz = res[2 * r + 1];
  const float c = R.cosrot[r], sn = R.sinrot[r];
  const float cx = c * px - sn * pz, cz = sn * px + c * pz;
  const float hl = R.xir[i * R.nrec + r] * R.gammar[j * R.nrec + r];
  const size_t g = (size_t)R.ibool[(size_t)R.ispec[r] * NGLL2 + p] * ps;
  atomicAdd(&D[2 * g], hl * cx);
  atomicAdd(&D[2 * g + 1], hl * cz);
}

// the Stacey traction's dependence on rho vp and rho vs at face point q, summed over the shots (point g of shot s at
// float2 g ps + s ss): gvp, gvs -= R~ . dB v'
__device__ __forceinline__ void stacey_gradient(const StaceyFaces& F, int q, int nshot, int ps, long ss,
                                                const float2* __restrict__ vpn, const float2* __restrict__ rb,
                                                float* __restrict__ gvp, float* __restrict__ gvs) {
  if (q >= F.nabs * NGLL) return;
  const int f = q / NGLL;
  const int ii = F.ij[2 * q], jj = F.ij[2 * q + 1];
  if (ii < 0 || jj < 0) return;  // corner point owned by the other edge
  const int g = F.ibool[(size_t)F.ispec[f] * NGLL2 + jj * NGLL + ii];
  const float nx = F.normal[2 * q], nz = F.normal[2 * q + 1], w = F.jacw[q];
  float sp = 0.f, sv = 0.f;
  for (int s = 0; s < nshot; s++) {
    const size_t o = (size_t)g * ps + (size_t)s * ss;
    const float2 v = vpn[o], b = rb[o];
    const float vn = nx * v.x + nz * v.y, bn = nx * b.x + nz * b.y;
    sp += w * vn * bn;
    sv += w * (v.x * b.x + v.y * b.y - vn * bn);
  }
  gvp[q] -= sp;
  gvs[q] -= sv;
}

}  // namespace sf2d
