// Exact discrete gradient of the L2 waveform misfit on the GPU: reverse mode of the elastic Newmark time loop
// with checkpointed forward recomputation.  No counterpart in the reference, whose SIMULATION_TYPE=3 path
// reconstructs the forward field backwards in time instead (src/specfem2D/compute_kernels.f90).
//
// One forward step n, as the reference's GPU sequence runs it (iterate_time.F90, compute_gpu_elastic.f90):
//     d_n = d + dt v + dt^2/2 a          v' = v + dt/2 a                      (predictor)
//     r_n = -K d_n - B v' + f_n                                               (forces, Stacey, sources)
//     a_n = W r_n                        v_n = v' + dt/2 a_n                  (W = rmass_inverse; corrector)
//     s_n = R d_n                                                             (seismograms)
// With the corrector deferred to the next step, the device fields after step n hold exactly (d_n, v', r_n): a
// checkpoint is a copy of them, and restoring one re-arms the pending corrector.
//
// Reverse step n, with (D, V, A) the cotangents of (d_n, v_n, a_n) and chi = 1/2 dt sum |s - o|^2:
//     D += R^T dt (s_n - o_n)
//     V' = V;  A += dt/2 V;  R~ = W A;   d chi/d M += -A r_n W^2           (k_adj_pointwise)
//     D += -K R~;  V' += -B R~                                              (the forward force and Stacey kernels)
//     d chi/d(kappa, mu) += -d a(d_n, R~)/d(kappa, mu);  d chi/d(rho vp, rho vs) += -R~ . dB v'   (k_grad_*)
//     V = V' + dt D;  A = dt/2 V' + dt^2/2 D                                 (folded into the next k_adj_pointwise)
// K and B are symmetric, so their transposes are the forward kernels themselves.  Gradients accumulate in FP32
// over one checkpoint segment and are added into FP64 totals at its end.
//
// A shot batch (batch.hip) runs the same sweep for all its shots at once: states, adjoint fields and residuals
// carry a shot dimension, while the gradient accumulators hold the sum over shots; the kernels that touch the
// accumulators loop over the shots, so each accumulator is read and written once per step for the batch.
#include <algorithm>

#include "sf2d_device.h"
#include "sf2d_mesh.h"
#include "specfem2d_gpu_ext.h"

namespace sf2d {

struct GradState {
  int nstep = 0, chunk = 0, nckpt = 0, nrec = 0, nshot = 1, batch = 0;
  size_t n2 = 0, ne = 0, nf = 0;
  long stride = 0;        // float2 between shots (shot-major: >= nglob; shot-minor: 1)
  int ps = 1;             // float2 between points (shot-minor: nshot)
  size_t nfield = 0;      // floats of one field over all shots
  float *fd = nullptr, *fv = nullptr, *fa = nullptr;  // the forward fields that states are copied from
  float* ckpt = nullptr;  // [nckpt][3][nfield]: (d, v', r) after steps chunk, 2 chunk, ...
  float* seg = nullptr;   // [chunk][3][nfield]: states of the segment being reversed
  float *D = nullptr, *Vb = nullptr, *Rb = nullptr;  // [nfield]
  float *gk32 = nullptr, *gm32 = nullptr, *pm32 = nullptr, *gvp32 = nullptr, *gvs32 = nullptr;
  double *gk = nullptr, *gm = nullptr, *pm = nullptr, *gvp = nullptr, *gvs = nullptr;
  float* res = nullptr;   // [nstep][nshot][nrec][2] = dt (s - o)
  // the fused sweep (handles with towers, shot-major fields): boundary terms of the recomputed steps [nfield], zero between
  // them, and the chains' row records with the points that each owns
  int fused = 0;
  float* acc = nullptr;
  int4* rows = nullptr;
  // R~ of the last nrb steps, Rb in a ring of nrb fields; the current step's is in slot rb_at.  npend steps, the first with
  // the forward state in segment slot pend_slot and R~ in ring slot pend_rb, wait for their strain products
  int nrb = 1, rb_at = 0, npend = 0, pend_slot = 0, pend_rb = 0;
  // the chain rule to (rho, vp, vs): model [3][ne] and Jacobian [ne] in the caller's element order, on the device or, where
  // that has little memory left, on the host
  double* model = nullptr;
  float* jac = nullptr;
  std::vector<double> h_model;
  std::vector<float> h_jac;
};

namespace {

constexpr int GT = 256;   // threads per workgroup
constexpr int RING = 4;   // steps per launch of k_grad_chain

constexpr int GEPB = 10;  // elements per workgroup in k_grad_elastic

// fields of shot s hold point g at float2 g + s ss (shot-major batches and single shots); one thread per point,
// both components at once, the shots four at a time so that twelve loads are in flight per thread
__device__ __forceinline__ void adj_point(int first, float dt, float dto2, float h, float2 w, float2 vb, float2 db,
                                          float2 rr, float2& v_out, float2& r_out, float2& dm) {
  float2 v = make_float2(0.f, 0.f), a = make_float2(0.f, 0.f);
  if (!first) {  // state cotangents of the step after this one
    v.x = vb.x + dt * db.x;
    v.y = vb.y + dt * db.y;
    a.x = dto2 * vb.x + h * db.x;
    a.y = dto2 * vb.y + h * db.y;
  }
  a.x = a.x + dto2 * v.x;
  a.y = a.y + dto2 * v.y;
  v_out = v;
  r_out = make_float2(w.x * a.x, w.y * a.y);
  dm.x += a.x * rr.x * w.x * w.x;
  dm.y += a.y * rr.y * w.y * w.y;
}

__global__ __launch_bounds__(GT) void k_adj_pointwise(int first, int npts, int nshot, long ss, float dt, float dto2,
                                                      float h, const float2* __restrict__ D, float2* __restrict__ Vb,
                                                      float2* __restrict__ Rb, const float* __restrict__ rmx,
                                                      const float* __restrict__ rmz, const float2* __restrict__ r,
                                                      float2* __restrict__ pm) {
  constexpr int U = 4;
  for (int g = blockIdx.x * blockDim.x + threadIdx.x; g < npts; g += gridDim.x * blockDim.x) {
    const float2 w = make_float2(rmx[g], rmz[g]);
    float2 dm = make_float2(0.f, 0.f);
    int s = 0;
    for (; s + U <= nshot; s += U) {
      float2 vb[U], db[U], rr[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const size_t q = (size_t)g + (size_t)(s + u) * ss;
        vb[u] = first ? make_float2(0.f, 0.f) : Vb[q];
        db[u] = first ? make_float2(0.f, 0.f) : D[q];
        rr[u] = r[q];
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const size_t q = (size_t)g + (size_t)(s + u) * ss;
        float2 vo, ro;
        adj_point(first, dt, dto2, h, w, vb[u], db[u], rr[u], vo, ro, dm);
        Vb[q] = vo;
        Rb[q] = ro;
      }
    }
    for (; s < nshot; s++) {
      const size_t q = (size_t)g + (size_t)s * ss;
      float2 vo, ro;
      adj_point(first, dt, dto2, h, w, first ? make_float2(0.f, 0.f) : Vb[q], first ? make_float2(0.f, 0.f) : D[q],
                r[q], vo, ro, dm);
      Vb[q] = vo;
      Rb[q] = ro;
    }
    float2 p = pm[g];
    p.x -= dm.x;
    p.y -= dm.y;
    pm[g] = p;
  }
}

// residual injection; shot blockIdx.y (residuals [nshot][nrec][2] of this step; D point g of shot s at float2
// g ps + s ss)
__global__ __launch_bounds__(64) void k_adj_receivers(const ReceiverSet R, const float* __restrict__ res,
                                                      float* __restrict__ D, int ps, long ss) {
  adjoint_receiver(R, blockIdx.x, threadIdx.x, res + (size_t)blockIdx.y * 2 * R.nrec, D + (size_t)2 * blockIdx.y * ss, ps);
}

// strain products of the forward displacement d_n and the adjoint force R~ at every element point, summed over
// the shots (point g of shot s at float2 g ps + s ss)
__global__ __launch_bounds__(GT) void k_grad_elastic(int nelem, int nshot, int ps, long ss, const int* __restrict__ ibool,
                                                     const float* __restrict__ xix, const float* __restrict__ xiz,
                                                     const float* __restrict__ gammax, const float* __restrict__ gammaz,
                                                     const float2* __restrict__ dn, const float2* __restrict__ rb,
                                                     float* __restrict__ gk, float* __restrict__ gm, const Basis basis) {
  __shared__ float s_hp[NGLL2];
  __shared__ float2 s_d[GT], s_b[GT];
  const int tid = threadIdx.x;
  if (tid < NGLL2) s_hp[tid] = basis.hp[tid];
  const int le = tid / NGLL2, p = tid - le * NGLL2, i = p % NGLL, j = p / NGLL;
  const int e = blockIdx.x * GEPB + le;
  const bool active = le < GEPB && e < nelem;
  const size_t l = (size_t)e * NGLL2 + p;
  const int g = active ? ibool[l] : 0;
  float X = 0.f, Z = 0.f, G = 0.f, H = 0.f;
  if (active) {
    X = xix[l];
    Z = xiz[l];
    G = gammax[l];
    H = gammaz[l];
  }
  const int base = le * NGLL2;
  const float wij = basis.w[i] * basis.w[j];  // read once, not per shot
  float sk = 0.f, sm = 0.f;
  // the next shot's two values are loaded while the current one is computed
  float2 dnext = make_float2(0.f, 0.f), bnext = dnext;
  if (active) {
    dnext = dn[(size_t)g * ps];
    bnext = rb[(size_t)g * ps];
  }
  for (int s = 0; s < nshot; s++) {
    if (s > 0) __syncthreads();  // the previous shot's LDS reads are done
    if (active) {
      s_d[tid] = dnext;
      s_b[tid] = bnext;
    }
    __syncthreads();
    if (active && s + 1 < nshot) {
      const size_t q = (size_t)g * ps + (size_t)(s + 1) * ss;
      dnext = dn[q];
      bnext = rb[q];
    }
    if (active) {
      float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < NGLL; k++) {
        const float hi = s_hp[i * NGLL + k], hj = s_hp[j * NGLL + k];
        const float2 dr = s_d[base + j * NGLL + k], dc = s_d[base + k * NGLL + i];
        const float2 br = s_b[base + j * NGLL + k], bc = s_b[base + k * NGLL + i];
        a[0] += dr.x * hi; a[1] += dr.y * hi; a[2] += dc.x * hj; a[3] += dc.y * hj;
        a[4] += br.x * hi; a[5] += br.y * hi; a[6] += bc.x * hj; a[7] += bc.y * hj;
      }
      const float ux = a[0] * X + a[2] * G, uxz = a[0] * Z + a[2] * H, uzx = a[1] * X + a[3] * G, uz = a[1] * Z + a[3] * H;
      const float wx = a[4] * X + a[6] * G, wxz = a[4] * Z + a[6] * H, wzx = a[5] * X + a[7] * G, wz = a[5] * Z + a[7] * H;
      const float wj = wij / (X * H - G * Z);
      sk += wj * (ux + uz) * (wx + wz);
      sm += wj * (ux * wx + uz * wz - ux * wz - uz * wx + (uxz + uzx) * (wxz + wzx));
    }
  }
  if (!active) return;
  gk[l] -= sk;
  gm[l] -= sm;
}

__global__ __launch_bounds__(64) void k_grad_stacey(const StaceyFaces F, int nshot, int ps, long ss,
                                                    const float2* __restrict__ vpn, const float2* __restrict__ rb,
                                                    float* __restrict__ gvp, float* __restrict__ gvs) {
  stacey_gradient(F, blockIdx.x * blockDim.x + threadIdx.x, nshot, ps, ss, vpn, rb, gvp, gvs);
}

// Shot-minor batches (nshot = 2^lshift values per point, at most 64): the same two reverse-sweep kernels with the
// shots in the lanes, so that every access is to consecutive values and the sum over the shots is a reduction
// across lanes.
// k_adj_pointwise over the flat points x shots x components entries; lanes of one (point, component) are 2 apart
__global__ __launch_bounds__(GT) void k_adj_pointwise_minor(int first, long n, int lshift, float dt, float dto2,
                                                            float h, const float* __restrict__ D,
                                                            float* __restrict__ Vb, float* __restrict__ Rb,
                                                            const float* __restrict__ rmx,
                                                            const float* __restrict__ rmz,
                                                            const float* __restrict__ r, float* __restrict__ pm) {
  const long stride = (long)gridDim.x * blockDim.x;  // a multiple of 64: groups of 2 nshot lanes stay together
  for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride) {
    const long g = k >> (lshift + 1);
    const int c = (int)(k & 1);
    const float w = c ? rmz[g] : rmx[g];
    float v = 0.f, a = 0.f;
    if (!first) {
      const float vb = Vb[k], db = D[k];
      v = vb + dt * db;
      a = dto2 * vb + h * db;
    }
    a = a + dto2 * v;
    Vb[k] = v;
    Rb[k] = w * a;
    float dm = a * r[k] * w * w;
    for (int o = 2; o < (2 << lshift); o <<= 1) dm += __shfl_xor(dm, o, 64);
    if (((k >> 1) & ((1 << lshift) - 1)) == 0) pm[2 * g + c] -= dm;
  }
}

// k_grad_elastic with lane = shot: a wave takes 64 / 2^lshift elements; each lane stages its element's two fields in
// lane-private LDS and the strain products of the 2^lshift lanes of an element are summed by shuffles
__global__ __launch_bounds__(64) void k_grad_elastic_minor(int nelem, int nshot, int lshift,
                                                           const int* __restrict__ ibool,
                                                           const float4* __restrict__ geom,
                                                           const float2* __restrict__ dn,
                                                           const float2* __restrict__ rb, float* __restrict__ gk,
                                                           float* __restrict__ gm, const Basis basis) {
  __shared__ float2 s_d[NGLL2][64], s_b[NGLL2][64];
  const int lane = threadIdx.x;
  const int per_wave = 64 >> lshift;
  const int wave = blockIdx.x;
  if (wave * per_wave >= nelem) return;  // uniform
  const int e = wave * per_wave + (lane >> lshift);
  const int s = lane & ((1 << lshift) - 1);
  const bool live = e < nelem && s < nshot;
  const unsigned ec = (unsigned)min(e, nelem - 1);
  const unsigned sh = (unsigned)min(s, nshot - 1);
  const unsigned ps = 1u << lshift;
#pragma unroll
  for (int p = 0; p < NGLL2; p++) {
    const unsigned g = (unsigned)ld_off(ibool, 4u * (ec * NGLL2 + p));
    s_d[p][lane] = ld_off(dn, 8u * (g * ps + sh));
    s_b[p][lane] = ld_off(rb, 8u * (g * ps + sh));
  }
#pragma unroll
  for (int j = 0; j < NGLL; j++) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NGLL; i++) {
      float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < NGLL; k++) {
        const float hi = basis.hp[i * NGLL + k], hj = basis.hp[j * NGLL + k];
        const float2 dr = s_d[j * NGLL + k][lane], dc = s_d[k * NGLL + i][lane];
        const float2 br = s_b[j * NGLL + k][lane], bc = s_b[k * NGLL + i][lane];
        a[0] += dr.x * hi; a[1] += dr.y * hi; a[2] += dc.x * hj; a[3] += dc.y * hj;
        a[4] += br.x * hi; a[5] += br.y * hi; a[6] += bc.x * hj; a[7] += bc.y * hj;
      }
      const unsigned l = ec * NGLL2 + j * NGLL + i;
      const float4 gp = ld_off(geom, 16u * l);
      const float X = gp.x, Z = gp.y, G = gp.z, H = gp.w;
      const float ux = a[0] * X + a[2] * G, uxz = a[0] * Z + a[2] * H, uzx = a[1] * X + a[3] * G, uz = a[1] * Z + a[3] * H;
      const float wx = a[4] * X + a[6] * G, wxz = a[4] * Z + a[6] * H, wzx = a[5] * X + a[7] * G, wz = a[5] * Z + a[7] * H;
      const float wj = basis.w[i] * basis.w[j] / (X * H - G * Z);
      float sk = live ? wj * (ux + uz) * (wx + wz) : 0.f;
      float sm = live ? wj * (ux * wx + uz * wz - ux * wz - uz * wx + (uxz + uzx) * (wxz + wzx)) : 0.f;
      for (int o = 1; o < (1 << lshift); o <<= 1) {
        sk += __shfl_xor(sk, o, 64);
        sm += __shfl_xor(sm, o, 64);
      }
      if (s == 0 && e < nelem) {
        gk[l] -= sk;
        gm[l] -= sm;
      }
    }
  }
}

// k_grad_elastic over chains, one wave per chain with lane 5 k + i holding column i of element k, for the fused reverse
// sweep: both fields' columns stay in registers, their rows pass through LDS, and the accumulators gk, gm lie in lane order
// (point (k, i, j) of the chain at e0 at e0 * 25 + j * 5 ne + 5 k + i) so that a wave reads and writes whole lines.  It
// also adds each point's mass term, pm -= R~ r W, where the chain owns the point (rows: masks of owned points).
// GEO as in tower.hip: 0 rectangles, 1 affine elements, 2 geometry per point.
// One launch takes nstep reverse steps: step t's fields are dn - t * state, rn - t * state and slot (rb0 + t) mod nrb of rb.
// Bound by HBM and L2, half of it the accumulators, read and written once a launch: 400 x 200
// elements 27 us for one step, 45 us for four; 8 shots of 300 x 150 46 and 145.
template <int GEO>
__global__ __launch_bounds__(64) void k_grad_chain(int nchain, int nstep, long state, int rb0, int nrb, long field,
                                                   int nshot, long ss, const int4* __restrict__ desc,
                                                   const int4* __restrict__ rows, const int* __restrict__ ends,
                                                   const float4* __restrict__ geom, const float4* __restrict__ geom_elem,
                                                   const float2* __restrict__ dn, const float2* __restrict__ rb,
                                                   const float2* __restrict__ rn, const float* __restrict__ rmx,
                                                   const float* __restrict__ rmz, float* __restrict__ gk,
                                                   float* __restrict__ gm, float2* __restrict__ pm, const Basis basis) {
  __shared__ float4 s_t[NGLL * 64 + 1];
  const int per = gridDim.x / NXCD;  // XCD-contiguous blocks of chains
  const int q = (blockIdx.x % NXCD) * per + blockIdx.x / NXCD;
  if (q >= nchain) return;  // uniform over the wave
  const int4 pd = desc[q];
  const int e0 = pd.x, ne = pd.w & 0xf;
  const int lane = threadIdx.x;
  const int k = min(lane / NGLL, Mesh::CHAIN_ELEMS);
  const int i = lane % NGLL;
  const int kk = min(k, ne - 1);
  const int x = 4 * kk + i;
  const bool active = lane / NGLL < ne;
  const bool writer = active && (i < NGLL - 1 || k == ne - 1);
  unsigned off[NGLL];
  bool own[NGLL];
#pragma unroll
  for (int j = 0; j < NGLL; j++) {
    const int4 r = rows[q * NGLL + j];
    off[j] = 8u * (unsigned)(x == 0 ? r.y : x == 4 * ne ? ends[q * NGLL + j] : r.x + x);
    const unsigned bits = x < 32 ? (unsigned)r.z >> x : (unsigned)r.w >> (x - 32);
    own[j] = writer && (bits & 1u);
  }
  float hpi[NGLL];
#pragma unroll
  for (int m = 0; m < NGLL; m++) hpi[m] = basis.hp[i * NGLL + m];
  float4 ge = make_float4(0.f, 0.f, 0.f, 0.f);
  if (GEO < 2) ge = geom_elem[e0 + kk];
  geom = at_element(geom, e0);
  const float4* const el = s_t + NGLL * k;
  float sk[NGLL], sm[NGLL];
  float2 dm[NGLL];
#pragma unroll
  for (int j = 0; j < NGLL; j++) {
    sk[j] = sm[j] = 0.f;
    dm[j] = make_float2(0.f, 0.f);
  }
  float2 d[NGLL], b[NGLL], r[NGLL];
  int step = 0, shot = 0;  // of the fields loaded next
  auto load = [&]() {
    const int slot = rb0 + step < nrb ? rb0 + step : rb0 + step - nrb;
    const long at = shot * ss - step * state, bt = shot * ss + slot * field;
#pragma unroll
    for (int j = 0; j < NGLL; j++) {
      d[j] = ld_off(dn + at, off[j]);
      b[j] = ld_off(rb + bt, off[j]);
      r[j] = own[j] ? ld_off(rn + at, off[j]) : make_float2(0.f, 0.f);
    }
    if (++shot == nshot) {
      shot = 0;
      step++;
    }
  };
  load();
  const int n = nstep * nshot;
  for (int s = 0; s < n; s++) {
    float4 u[NGLL];
#pragma unroll
    for (int j = 0; j < NGLL; j++) {
      u[j] = make_float4(d[j].x, d[j].y, b[j].x, b[j].y);
      dm[j].x += b[j].x * r[j].x;
      dm[j].y += b[j].y * r[j].y;
    }
    if (s + 1 < n) load();  // the next shot's or step's values are in flight while this one is computed
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < NGLL; j++) s_t[j * 64 + lane] = u[j];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < NGLL; j++) {
      float4 xi = make_float4(0.f, 0.f, 0.f, 0.f), ga = xi;
#pragma unroll
      for (int m = 0; m < NGLL; m++) {
        const float4 e = el[j * 64 + m];
        const float h = basis.hp[j * NGLL + m];
        xi.x += e.x * hpi[m];
        xi.y += e.y * hpi[m];
        xi.z += e.z * hpi[m];
        xi.w += e.w * hpi[m];
        ga.x += u[m].x * h;
        ga.y += u[m].y * h;
        ga.z += u[m].z * h;
        ga.w += u[m].w * h;
      }
      float4 gp = ge;
      if (GEO == 2) gp = ld_off(geom, 16u * (unsigned)(kk * NGLL2 + j * NGLL + i));
      const float X = gp.x, Z = GEO ? gp.y : 0.f, G = GEO ? gp.z : 0.f, H = gp.w;
      const float ux = xi.x * X + ga.x * G, uxz = xi.x * Z + ga.x * H, uzx = xi.y * X + ga.y * G, uz = xi.y * Z + ga.y * H;
      const float wx = xi.z * X + ga.z * G, wxz = xi.z * Z + ga.z * H, wzx = xi.w * X + ga.w * G, wz = xi.w * Z + ga.w * H;
      sk[j] += (ux + uz) * (wx + wz);
      sm[j] += ux * wx + uz * wz - ux * wz - uz * wx + (uxz + uzx) * (wxz + wzx);
    }
  }
  unsigned l = (unsigned)e0 * NGLL2 + (unsigned)lane;
#pragma unroll
  for (int j = 0; j < NGLL; j++) {
    float4 gp = ge;
    if (GEO == 2) gp = ld_off(geom, 16u * (unsigned)(kk * NGLL2 + j * NGLL + i));
    const float X = gp.x, Z = GEO ? gp.y : 0.f, G = GEO ? gp.z : 0.f, H = gp.w;
    const float wj = basis.w[i] * basis.w[j] / (X * H - G * Z);
    if (active) {
      gk[l] -= wj * sk[j];
      gm[l] -= wj * sm[j];
    }
    l += (unsigned)(NGLL * ne);
    if (own[j]) {
      const unsigned g = off[j] / 8u;
      float2 p = pm[g];
      p.x -= dm[j].x * rmx[g];
      p.y -= dm[j].y * rmz[g];
      pm[g] = p;
    }
  }
}

__global__ __launch_bounds__(GT) void k_flush64(size_t n, float* __restrict__ a32, double* __restrict__ a64) {
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < n; k += (size_t)gridDim.x * blockDim.x) {
    a64[k] += (double)a32[k];
    a32[k] = 0.f;
  }
}

// The chain rule from the accumulators to (rho, vp, vs) in 64 bits, one thread per element point in the caller's order:
// mu = rho vs^2, kappa = rho vp^2 - mu, and the mass term M_c(g) = sum w_i w_j J rho.  For the ne element points of a range
// of elements, of which where, jac, model (components mstride apart) and out hold the range alone.  where[e]: {element
// position, first accumulator word, words from one j to the next, -}.  out: [3][ne] gradient, then (parts) [5][ne]
// d chi / d (kappa, mu, rho through the mass, rho vp, rho vs).  Bound by its reads and writes, 100 bytes a point; on the host
// the same loops, with their arrays, took half of a gradient (400 x 200 elements: 30 of 59 ms).
__global__ __launch_bounds__(GT) void k_grad_model(long ne, long mstride, const int4* __restrict__ where,
                                                   const int* __restrict__ ibool,
                                                   const double* __restrict__ gk, const double* __restrict__ gm,
                                                   const double* __restrict__ pm, const double* __restrict__ model,
                                                   const float* __restrict__ jac, double* __restrict__ out, int parts,
                                                   const Basis basis) {
  const long l = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= ne) return;
  const int e = (int)(l / NGLL2), p = (int)(l - (long)e * NGLL2), i = p % NGLL, j = p / NGLL;
  const int4 q = where[e];
  const size_t at = (size_t)q.y + (size_t)j * q.z + i;
  const size_t g = (size_t)ibool[(size_t)q.x * NGLL2 + p];
  const double a = gk[at], b = gm[at];
  const double w = (double)basis.w[i] * (double)basis.w[j] * (double)jac[l];
  const double r = w * (pm[2 * g] + pm[2 * g + 1]);
  const double rho = model[l], vp = model[mstride + l], vs = model[2 * mstride + l];
  out[l] = a * (vp * vp - vs * vs) + b * vs * vs + r;
  out[ne + l] = a * 2.0 * rho * vp;
  out[2 * ne + l] = -a * 2.0 * rho * vs + b * 2.0 * rho * vs;
  if (parts) {
    out[3 * ne + l] = a;
    out[4 * ne + l] = b;
    out[5 * ne + l] = r;
    out[6 * ne + l] = 0.0;
    out[7 * ne + l] = 0.0;
  }
}

// the Stacey traction's part and its Newmark mass term T_c = dt/2 w [rho_vp (nx+nz) n_c + rho_vs (1 - (nx+nz) n_c)], one
// thread per face point, of the faces in elements e0 .. e0 + ne / 25 - 1; ispec_of_pos: the caller's element at each position
__global__ __launch_bounds__(64) void k_grad_model_stacey(const StaceyFaces F, int e0, long ne, long mstride,
                                                          const int* __restrict__ ispec_of_pos,
                                                          const double* __restrict__ gvp, const double* __restrict__ gvs,
                                                          const double* __restrict__ pm,
                                                          const double* __restrict__ model, double dto2,
                                                          double* __restrict__ out, int parts) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= F.nabs * NGLL) return;
  const int ii = F.ij[2 * q], jj = F.ij[2 * q + 1];
  if (ii < 0 || jj < 0) return;
  const int pos = F.ispec[q / NGLL], p = jj * NGLL + ii;
  const size_t g = (size_t)F.ibool[(size_t)pos * NGLL2 + p];
  const long l = (long)(ispec_of_pos[pos] - e0) * NGLL2 + p;
  if (l < 0 || l >= ne) return;
  const double nx = F.normal[2 * q], nz = F.normal[2 * q + 1], w = F.jacw[q];
  const double sn = nx + nz, px = pm[2 * g], pz = pm[2 * g + 1];
  const double a = gvp[q] + w * dto2 * (px * sn * nx + pz * sn * nz);
  const double b = gvs[q] + w * dto2 * (px * (1.0 - sn * nx) + pz * (1.0 - sn * nz));
  const double rho = model[l], vp = model[mstride + l], vs = model[2 * mstride + l];
  // corner elements have two faces, hence atomics; two terms added to a third in either order differ in the last bit
  unsafeAtomicAdd(&out[l], a * vp + b * vs);
  unsafeAtomicAdd(&out[ne + l], a * rho);
  unsafeAtomicAdd(&out[2 * ne + l], b * rho);
  if (parts) {
    unsafeAtomicAdd(&out[6 * ne + l], a);
    unsafeAtomicAdd(&out[7 * ne + l], b);
  }
}

int grid_for(size_t n) { return (int)std::min<size_t>((n + GT - 1) / GT, 65536); }

GradState* need(Mesh* mp) {
  if (!mp->grad) fail("gradient buffers not prepared (sf2d_grad_prepare)");
  return mp->grad;
}

void copy_d2d(float* dst, const float* src, size_t n, hipStream_t s) {
  check_hip(hipMemcpyAsync(dst, src, n * sizeof(float), hipMemcpyDeviceToDevice, s), "gradient state copy");
}

// buffers for checkpoints every `chunk` steps, one segment of states and the accumulators, over the handle's
// own forward fields (batch = 0) or over its shot batch (batch = 1); returns the number of checkpoints
int grad_prepare(Mesh* mp, long* Mesh_pointer, int chunk, int nrec, int batch) {
  if (chunk < 1) fail("gradient: chunk %d < 1", chunk);
  if (nrec != mp->nrec_local) fail("gradient: %d receivers, the handle has %d", nrec, mp->nrec_local);
  if (GradState* old = mp->grad) {  // same layout as the buffers in place: keep them (repeated gradients)
    bool same = old->batch == batch && old->chunk == std::min(chunk, mp->nstep) && old->nstep == mp->nstep &&
                old->nrec == nrec;
    if (same && batch) {
      float *d, *v, *a;
      int ns, ps;
      long st;
      batch_fields(mp, &d, &v, &a, &ns, &st, &ps);
      same = old->fd == d && old->nshot == ns && old->stride == st && old->ps == ps;
    }
    if (same) return old->nckpt;
    sf2d_grad_release(Mesh_pointer);
  }
  GradState* G = new GradState();
  G->nstep = mp->nstep;
  G->chunk = std::min(chunk, mp->nstep);
  G->nckpt = (mp->nstep - 1) / G->chunk;
  G->nrec = nrec;
  G->n2 = (size_t)2 * mp->nglob;
  G->ne = (size_t)mp->nspec * NGLL2;
  G->nf = (size_t)mp->num_abs * NGLL;
  G->batch = batch;
  if (batch) {
    batch_fields(mp, &G->fd, &G->fv, &G->fa, &G->nshot, &G->stride, &G->ps);
  } else {
    G->fd = mp->d_displ;
    G->fv = mp->d_veloc;
    G->fa = mp->d_accel;
    G->nshot = 1;
    G->stride = mp->nglob;
    G->ps = 1;
  }
  G->nfield = G->ps > 1 ? (size_t)2 * mp->nglob * G->nshot : (size_t)2 * G->stride * G->nshot;
  if (G->ps > 1 && (G->ps > 64 || (G->ps & (G->ps - 1)) || !mp->d_geom))
    fail("gradient: shot-minor batches need a power of two of at most 64 shots and the patch assembly");
  const size_t states = (size_t)std::max(1, G->nckpt) + G->chunk;
  if (states * 3 * G->nfield * sizeof(float) > ((size_t)240 << 30))
    fail("gradient: %zu states of %d shots exceed 240 GiB; use a longer chunk or fewer shots", states, G->nshot);
  // the states before a faster step
  if ((states + 1) * 3 * G->nfield * sizeof(float) + (3 * G->ne + 2 * G->n2) * sizeof(double) > spare_memory()) tower_release(mp);
  G->ckpt = device_alloc<float>(3 * G->nfield * std::max(1, G->nckpt));  // written before they are read
  G->seg = device_alloc<float>(3 * G->nfield * G->chunk);
  G->D = device_zeros<float>(G->nfield);
  G->Vb = device_zeros<float>(G->nfield);
  G->Rb = device_zeros<float>(G->nfield);
  G->gk32 = device_zeros<float>(G->ne);
  G->gm32 = device_zeros<float>(G->ne);
  G->pm32 = device_zeros<float>(G->n2);
  G->gvp32 = device_zeros<float>(std::max<size_t>(1, G->nf));
  G->gvs32 = device_zeros<float>(std::max<size_t>(1, G->nf));
  G->gk = device_zeros<double>(G->ne);
  G->gm = device_zeros<double>(G->ne);
  G->pm = device_zeros<double>(G->n2);
  G->gvp = device_zeros<double>(std::max<size_t>(1, G->nf));
  G->gvs = device_zeros<double>(std::max<size_t>(1, G->nf));
  G->res = device_zeros<float>((size_t)std::max(1, nrec) * 2 * G->nshot * mp->nstep);
  mp->grad = G;
  mp->grad_batch = batch;
  return G->nckpt;
}

// the strain products of the steps that wait for them
void flush_pending(Mesh* mp, GradState* G) {
  if (G->npend == 0) return;
  using K = decltype(&k_grad_chain<0>);
  const K kern[3] = {k_grad_chain<0>, k_grad_chain<1>, k_grad_chain<2>};
  const int geo = mp->rect ? 0 : (!mp->no_affine && mp->n_affine == mp->nspec) ? 1 : 2;
  const long field = (long)(G->nfield / 2);
  const float2* dn = (const float2*)(G->seg + (size_t)G->pend_slot * 3 * G->nfield);
  hipLaunchKernelGGL(kern[geo], dim3((mp->npatch + NXCD - 1) / NXCD * NXCD), dim3(64), 0, mp->stream, mp->npatch, G->npend,
                     3 * field, G->pend_rb, G->nrb, field, G->nshot, G->stride, mp->d_patch_desc, G->rows, mp->d_col_ends,
                     mp->d_geom, mp->d_geom_elem, dn, (const float2*)G->Rb, dn + 2 * field, mp->d_rmassx, mp->d_rmassz,
                     G->gk32, G->gm32, (float2*)G->pm32, mp->basis);
  check_hip(hipGetLastError(), "k_grad_chain launch");
  G->npend = 0;
}

// whether the sweep runs on towers, and what that needs: with a tower per chain stack, shot-major fields and neither a
// CPML layer nor attenuation (which gradients refuse)
void choose_sweep(Mesh* mp, GradState* G) {
  G->rb_at = G->npend = 0;
  G->fused = G->ps == 1 && tower_takes(mp, G->nshot) && !mp->pml && !mp->attenuation;
  if (!G->fused || G->rows) return;
  // the boundary terms' field has to fit, and a ring of R~ has to leave most of the memory free: steps to take at once
  const size_t free_bytes = spare_memory();
  const size_t bytes = G->nfield * sizeof(float);
  if (free_bytes < 2 * bytes) {
    G->fused = 0;
    return;
  }
  if (free_bytes > 8 * RING * bytes) {
    device_free(G->Rb);
    G->Rb = device_zeros<float>(RING * G->nfield);
    G->nrb = RING;
  }
  const int n = mp->npatch;
  std::vector<int4> rows(mp->h_col_rows);
  std::vector<char> seen((size_t)mp->nglob, 0);
  for (int q = 0; q < n; q++) {
    const int ne = mp->h_patch_desc[4 * q + 3] & 0xf;
    for (int j = 0; j < NGLL; j++) {
      int4& r = rows[(size_t)q * NGLL + j];
      unsigned long long mask = 0ull;
      for (int x = 0; x <= 4 * ne; x++) {
        char& s = seen[x == 0 ? r.y : x == 4 * ne ? mp->h_col_ends[(size_t)q * NGLL + j] : r.x + x];
        if (!s) mask |= 1ull << x;
        s = 1;
      }
      r.z = (int)(unsigned)(mask & 0xffffffffull);
      r.w = (int)(unsigned)(mask >> 32);
    }
  }
  G->rows = device_copy(rows.data(), rows.size());
  G->acc = device_zeros<float>(G->nfield);
}

// where each caller element's accumulators lie: {element position, first word, words from one j to the next, -}, element
// position by position or, in a fused sweep, in the lane order of the chain at e0
std::vector<int4> accumulator_places(const Mesh* mp, const GradState* G) {
  std::vector<int4> where((size_t)mp->nspec);
  for (int e = 0; e < mp->nspec; e++) {
    const int pos = mp->pos_of_ispec[e];
    where[e] = make_int4(pos, pos * NGLL2, NGLL, 0);
  }
  if (G->fused)
    for (int q = 0; q < mp->npatch; q++) {
      const int e0 = mp->h_patch_desc[4 * q], n = mp->h_patch_desc[4 * q + 3] & 0xf;
      for (int k = 0; k < n; k++) where[mp->ispec_of_pos[e0 + k]] = make_int4(e0 + k, e0 * NGLL2 + NGLL * k, NGLL * n, 0);
    }
  return where;
}

}  // namespace

float* grad_checkpoint_inputs(Mesh* mp, int slot) {
  GradState* G = need(mp);
  if (slot < 0 || slot >= G->nckpt) fail("gradient checkpoint %d outside 0..%d", slot, G->nckpt - 1);
  float* dst = G->ckpt + (size_t)slot * 3 * G->nfield;
  copy_d2d(dst, G->fd, G->nfield, mp->stream);
  copy_d2d(dst + G->nfield, G->fv, G->nfield, mp->stream);
  return dst + 2 * G->nfield;
}

}  // namespace sf2d

using namespace sf2d;

extern "C" {

int sf2d_grad_prepare(long* Mesh_pointer, int chunk, int nrec) {
  Mesh* mp = handle(Mesh_pointer);
  if (!mp->sorted) fail("sf2d_grad_prepare: prepare_fields_elastic_device was not called");
  if (mp->nspec_acoustic > 0) fail("sf2d_grad_prepare: gradients of meshes with fluid elements are not supported");
  return grad_prepare(mp, Mesh_pointer, chunk, nrec, 0);
}

int sf2d_batch_grad_prepare(long* Mesh_pointer, int chunk) {
  Mesh* mp = handle(Mesh_pointer);
  if (!mp->batch) fail("sf2d_batch_grad_prepare: shot batch not prepared (sf2d_batch_prepare)");
  return grad_prepare(mp, Mesh_pointer, chunk, mp->nrec_local, 1);
}

void sf2d_grad_release(long* Mesh_pointer) {
  Mesh* mp = handle(Mesh_pointer);
  GradState* G = mp->grad;
  if (!G) return;
  check_hip(hipStreamSynchronize(mp->stream), "sf2d_grad_release");
  for (float** p : {&G->ckpt, &G->seg, &G->D, &G->Vb, &G->Rb, &G->gk32, &G->gm32, &G->pm32, &G->gvp32, &G->gvs32,
                    &G->res, &G->acc})
    device_free(*p);
  device_free(G->rows);
  device_free(G->jac);
  for (double** p : {&G->gk, &G->gm, &G->pm, &G->gvp, &G->gvs, &G->model}) device_free(*p);
  delete G;
  mp->grad = nullptr;
  mp->grad_batch = 0;
}

// copies the forward fields (d_n, v', r_n) after a step into checkpoint (kind 0) or segment (kind 1) slot
void sf2d_grad_save_state(long* Mesh_pointer, int kind, int slot) {
  Mesh* mp = handle(Mesh_pointer);
  GradState* G = need(mp);
  const int nslot = kind == 0 ? G->nckpt : G->chunk;
  if (slot < 0 || slot >= nslot) fail("sf2d_grad_save_state: slot %d outside 0..%d", slot, nslot - 1);
  float* dst = (kind == 0 ? G->ckpt : G->seg) + (size_t)slot * 3 * G->nfield;
  copy_d2d(dst, G->fd, G->nfield, mp->stream);
  copy_d2d(dst + G->nfield, G->fv, G->nfield, mp->stream);
  copy_d2d(dst + 2 * G->nfield, G->fa, G->nfield, mp->stream);
}

// 1 when the sweep begun by sf2d_grad_begin_reverse recomputes with sf2d_grad_recompute_segment (always so for batches)
int sf2d_grad_fused(long* Mesh_pointer) { return need(handle(Mesh_pointer))->fused; }

// leaves the handle's own fields in the state of segment slot (the corrector of that step pending)
void sf2d_grad_load_segment(long* Mesh_pointer, int slot, float dto2) {
  Mesh* mp = handle(Mesh_pointer);
  GradState* G = need(mp);
  if (G->batch || slot < 0 || slot >= G->chunk) fail("sf2d_grad_load_segment: slot %d", slot);
  const float* src = G->seg + (size_t)slot * 3 * G->nfield;
  copy_d2d(G->fd, src, G->nfield, mp->stream);
  copy_d2d(G->fv, src + G->nfield, G->nfield, mp->stream);
  copy_d2d(G->fa, src + 2 * G->nfield, G->nfield, mp->stream);
  mp->pending_corrector[0] = 1;
  mp->pending_dto2[0] = dto2;
  mp->accel_partial = 0;
}

// restores checkpoint slot into the forward fields, with the corrector of that step pending (dto2 = dt/2)
void sf2d_grad_restore_checkpoint(long* Mesh_pointer, int slot, float dto2) {
  Mesh* mp = handle(Mesh_pointer);
  GradState* G = need(mp);
  if (slot < 0 || slot >= G->nckpt) fail("sf2d_grad_restore_checkpoint: slot %d outside 0..%d", slot, G->nckpt - 1);
  const float* src = G->ckpt + (size_t)slot * 3 * G->nfield;
  copy_d2d(G->fd, src, G->nfield, mp->stream);
  copy_d2d(G->fv, src + G->nfield, G->nfield, mp->stream);
  copy_d2d(G->fa, src + 2 * G->nfield, G->nfield, mp->stream);
  if (G->batch) {
    batch_set_pending(mp, dto2);
  } else {
    mp->pending_corrector[0] = 1;
    mp->pending_dto2[0] = dto2;
    mp->accel_partial = 0;
  }
}

// residuals dt (s - o) for all steps, [nstep][nshot][nrec][2]; zeroes the adjoint state and the accumulators
void sf2d_grad_begin_reverse(long* Mesh_pointer, const float* res) {
  Mesh* mp = handle(Mesh_pointer);
  GradState* G = need(mp);
  if (G->nrec > 0)
    check_hip(hipMemcpyAsync(G->res, res, sizeof(float) * 2 * G->nrec * G->nshot * G->nstep, hipMemcpyHostToDevice,
                             mp->stream),
              "residual H2D");
  choose_sweep(mp, G);
  for (float* p : {G->D, G->Vb}) check_hip(hipMemsetAsync(p, 0, G->nfield * sizeof(float), mp->stream), "zero");
  check_hip(hipMemsetAsync(G->Rb, 0, G->nrb * G->nfield * sizeof(float), mp->stream), "zero");
  check_hip(hipMemsetAsync(G->pm32, 0, G->n2 * sizeof(float), mp->stream), "zero");
  for (float* p : {G->gk32, G->gm32}) check_hip(hipMemsetAsync(p, 0, G->ne * sizeof(float), mp->stream), "zero");
  for (double* p : {G->gk, G->gm}) check_hip(hipMemsetAsync(p, 0, G->ne * sizeof(double), mp->stream), "zero");
  check_hip(hipMemsetAsync(G->pm, 0, G->n2 * sizeof(double), mp->stream), "zero");
  const size_t nf = std::max<size_t>(1, G->nf);
  for (float* p : {G->gvp32, G->gvs32}) check_hip(hipMemsetAsync(p, 0, nf * sizeof(float), mp->stream), "zero");
  for (double* p : {G->gvp, G->gvs}) check_hip(hipMemsetAsync(p, 0, nf * sizeof(double), mp->stream), "zero");
  check_hip(hipStreamSynchronize(mp->stream), "sf2d_grad_begin_reverse");
}

// reverse step n (1-based) from the states in segment slot (d_n, v', r_n); first = 1 for n = NSTEP
void sf2d_grad_reverse_step(long* Mesh_pointer, int n, int slot, int first, float dt) {
  Mesh* mp = handle(Mesh_pointer);
  GradState* G = need(mp);
  if (n < 1 || n > G->nstep) fail("sf2d_grad_reverse_step: step %d outside 1..%d", n, G->nstep);
  if (slot < 0 || slot >= G->chunk) fail("sf2d_grad_reverse_step: slot %d outside 0..%d", slot, G->chunk - 1);
  const float* dn = G->seg + (size_t)slot * 3 * G->nfield;
  const float* vpn = dn + G->nfield;
  const float* rn = dn + 2 * G->nfield;
  const float dto2 = (float)(0.5 * (double)dt), h = (float)(0.5 * (double)dt * (double)dt);
  const float* res = G->res + (size_t)(n - 1) * 2 * G->nrec * G->nshot;
  if (G->fused) {
    if (!mp->tower) fail("sf2d_grad_reverse_step: the materials changed during the sweep");
    // R~_n is complete: the previous step's update made it (zero at n = NSTEP)
    if (!first) {
      if (G->npend == 0) {
        G->pend_slot = slot;
        G->pend_rb = G->rb_at;
      }
      if (++G->npend == G->nrb) flush_pending(mp, G);
    }
    const int next = (G->rb_at + 1) % G->nrb;
    tower_step_adjoint(mp, G->Rb + G->rb_at * G->nfield, G->Rb + next * G->nfield, G->D, G->Vb, G->stride, G->nshot, res,
                       vpn, G->gvp32, G->gvs32, dt, h, dto2);
    G->rb_at = next;
    return;
  }
  int lshift = 0;
  while ((1 << lshift) < G->ps) lshift++;
  if (G->ps > 1)
    hipLaunchKernelGGL(k_adj_pointwise_minor, dim3(grid_for(G->nfield)), dim3(GT), 0, mp->stream, first,
                       (long)G->nfield, lshift, dt, dto2, h, G->D, G->Vb, G->Rb, mp->d_rmassx, mp->d_rmassz, rn,
                       G->pm32);
  else
    hipLaunchKernelGGL(k_adj_pointwise, dim3(grid_for(G->n2 / 2)), dim3(GT), 0, mp->stream, first, (int)(G->n2 / 2),
                       G->nshot, G->stride, dt, dto2, h, (const float2*)G->D, (float2*)G->Vb, (float2*)G->Rb,
                       mp->d_rmassx, mp->d_rmassz, (const float2*)rn, (float2*)G->pm32);
  if (G->nrec > 0)
    hipLaunchKernelGGL(k_adj_receivers, dim3(G->nrec, G->nshot), dim3(64), 0, mp->stream, receiver_set(mp),
                       res, G->D, G->ps, G->stride);
  apply_element_forces(mp, 0, G->Rb, G->D, G->nshot, G->stride, 0, G->ps);
  apply_element_forces(mp, 1, G->Rb, G->D, G->nshot, G->stride, 0, G->ps);
  if (mp->stacey && mp->num_abs > 0) {
    launch_stacey(mp, G->Rb, G->Vb, 0, G->nshot, G->stride, G->ps);
    hipLaunchKernelGGL(k_grad_stacey, dim3((mp->num_abs * NGLL + 63) / 64), dim3(64), 0, mp->stream,
                       stacey_faces(mp), G->nshot, G->ps, G->stride, (const float2*)vpn, (const float2*)G->Rb, G->gvp32,
                       G->gvs32);
  }
  if (G->ps > 1)
    hipLaunchKernelGGL(k_grad_elastic_minor, dim3((mp->nspec + (64 >> lshift) - 1) / (64 >> lshift)), dim3(64), 0,
                       mp->stream, mp->nspec, G->nshot, lshift, mp->d_ibool, mp->d_geom, (const float2*)dn,
                       (const float2*)G->Rb, G->gk32, G->gm32, mp->basis);
  else
    hipLaunchKernelGGL(k_grad_elastic, dim3((mp->nspec + GEPB - 1) / GEPB), dim3(GT), 0, mp->stream, mp->nspec,
                       G->nshot, G->ps, G->stride, mp->d_ibool, mp->d_xix, mp->d_xiz, mp->d_gammax, mp->d_gammaz,
                       (const float2*)dn, (const float2*)G->Rb, G->gk32, G->gm32, mp->basis);
  check_hip(hipGetLastError(), "sf2d_grad_reverse_step launch");
}

// recomputes steps n0+1 .. n1 straight into the segment slots, from checkpoint slot ckpt (the state after step n0) or
// from rest (ckpt = -1, n0 = 0); no state is copied.  Shot batches, and the handle's own fields in a fused sweep.
void sf2d_grad_recompute_segment(long* Mesh_pointer, int ckpt, int n0, int n1, float dt) {
  Mesh* mp = handle(Mesh_pointer);
  GradState* G = need(mp);
  if (!G->batch && !G->fused) fail("sf2d_grad_recompute_segment: neither a shot batch nor a fused sweep");
  if (n0 < 0 || n1 <= n0 || n1 > G->nstep || n1 - n0 > G->chunk)
    fail("sf2d_grad_recompute_segment: steps %d..%d (segments of at most %d)", n0 + 1, n1, G->chunk);
  if (ckpt < -1 || ckpt >= G->nckpt || (ckpt == -1) != (n0 == 0))
    fail("sf2d_grad_recompute_segment: checkpoint %d for a segment after step %d", ckpt, n0);
  const float dto2 = (float)(0.5 * (double)dt), h = (float)(0.5 * (double)dt * (double)dt);
  const float* src = ckpt < 0 ? nullptr : G->ckpt + (size_t)ckpt * 3 * G->nfield;
  if (G->fused) {
    if (!mp->tower) fail("sf2d_grad_recompute_segment: the materials changed during the sweep");
    if (!src) {  // the predictor of a state at rest is the state at rest
      for (int f = 0; f < 2; f++)
        check_hip(hipMemsetAsync(G->seg + f * G->nfield, 0, G->nfield * sizeof(float), mp->stream), "zero");
    } else {  // into the accelerations of slot 0 too, where the step's forces overwrite them
      launch_newmark_corrector_predictor_to(src, src + G->nfield, src + 2 * G->nfield, G->seg, G->seg + G->nfield,
                                            G->seg + 2 * G->nfield, mp->d_rmassx, mp->d_rmassz, mp->nglob, dto2, dt, h,
                                            dto2, mp->stream, G->nshot, G->stride, 1, 1);
    }
    for (int n = n0 + 1; n <= n1; n++) {
      float* at = G->seg + (size_t)(n - n0 - 1) * 3 * G->nfield;
      float* next = n < n1 ? at + 3 * G->nfield : at;
      tower_step_shots(mp, {at, at + G->nfield, next, next + G->nfield, at + 2 * G->nfield, G->acc, G->stride, G->nshot,
                            n < n1 ? 0 : 2, G->batch ? batch_source_shots(mp) : nullptr, nullptr, nullptr},
                       n, dt, h, dto2);
    }
    return;
  }
  for (int n = n0 + 1; n <= n1; n++) {
    float* dst = G->seg + (size_t)(n - n0 - 1) * 3 * G->nfield;
    batch_step_into(mp, n, src, src ? src + G->nfield : nullptr, src ? src + 2 * G->nfield : nullptr, dto2, dst,
                    dst + G->nfield, dst + 2 * G->nfield, dt, h, dto2);
    src = dst;
  }
}

// adds the FP32 segment accumulators into the FP64 totals
void sf2d_grad_flush(long* Mesh_pointer) {
  Mesh* mp = handle(Mesh_pointer);
  GradState* G = need(mp);
  flush_pending(mp, G);
  hipLaunchKernelGGL(k_flush64, dim3(grid_for(G->ne)), dim3(GT), 0, mp->stream, G->ne, G->gk32, G->gk);
  hipLaunchKernelGGL(k_flush64, dim3(grid_for(G->ne)), dim3(GT), 0, mp->stream, G->ne, G->gm32, G->gm);
  hipLaunchKernelGGL(k_flush64, dim3(grid_for(G->n2)), dim3(GT), 0, mp->stream, G->n2, G->pm32, G->pm);
  if (G->nf) {
    hipLaunchKernelGGL(k_flush64, dim3(grid_for(G->nf)), dim3(GT), 0, mp->stream, G->nf, G->gvp32, G->gvp);
    hipLaunchKernelGGL(k_flush64, dim3(grid_for(G->nf)), dim3(GT), 0, mp->stream, G->nf, G->gvs32, G->gvs);
  }
  check_hip(hipGetLastError(), "sf2d_grad_flush launch");
}

// FP64 totals in the caller's numbering: g_kappa, g_mu [nspec][25] (ispec order), d chi/d M [nglob][2],
// Stacey traction parts [nabs][5] (rho vp, rho vs)
void sf2d_grad_result(long* Mesh_pointer, double* gk, double* gm, double* pm, double* gvp, double* gvs) {
  Mesh* mp = handle(Mesh_pointer);
  GradState* G = need(mp);
  check_hip(hipStreamSynchronize(mp->stream), "sf2d_grad_result");
  std::vector<double> t(std::max(G->ne, G->n2));
  const std::vector<int4> where = accumulator_places(mp, G);
  auto elem = [&](const double* dev, double* out) {
    check_hip(hipMemcpy(t.data(), dev, G->ne * sizeof(double), hipMemcpyDeviceToHost), "gradient D2H");
    for (int e = 0; e < mp->nspec; e++)
      for (int p = 0; p < NGLL2; p++)
        out[(size_t)e * NGLL2 + p] = t[(size_t)where[e].y + (size_t)(p / NGLL) * where[e].z + p % NGLL];
  };
  elem(G->gk, gk);
  elem(G->gm, gm);
  check_hip(hipMemcpy(t.data(), G->pm, G->n2 * sizeof(double), hipMemcpyDeviceToHost), "gradient D2H");
  for (int g = 0; g < mp->nglob; g++) {
    const size_t id = mp->point_id.empty() ? (size_t)g : (size_t)mp->point_id[g];
    pm[2 * g] = t[2 * id];
    pm[2 * g + 1] = t[2 * id + 1];
  }
  if (G->nf) {
    check_hip(hipMemcpy(gvp, G->gvp, G->nf * sizeof(double), hipMemcpyDeviceToHost), "gradient D2H");
    check_hip(hipMemcpy(gvs, G->gvs, G->nf * sizeof(double), hipMemcpyDeviceToHost), "gradient D2H");
  }
}

// the model of the chain rule, after sf2d_grad_prepare and whenever the model changes: rho, vp, vs and the Jacobian
// [nspec][25] in ispec order.  It stays on the device where it takes an eighth of the spare memory at most: checkpoints are
// made to fill the card, and a gradient must not fail at its end.
void sf2d_grad_set_model(long* Mesh_pointer, const double* rho, const double* vp, const double* vs, const float* jacobian) {
  Mesh* mp = handle(Mesh_pointer);
  GradState* G = need(mp);
  const double* m[3] = {rho, vp, vs};
  if (!G->model && spare_memory() / 8 < G->ne * (3 * sizeof(double) + sizeof(float))) {
    G->h_model.resize(3 * G->ne);
    for (int k = 0; k < 3; k++) std::copy(m[k], m[k] + G->ne, G->h_model.begin() + k * G->ne);
    G->h_jac.assign(jacobian, jacobian + G->ne);
    return;
  }
  if (!G->model) {
    G->model = device_alloc<double>(3 * G->ne);
    G->jac = device_alloc<float>(G->ne);
  }
  for (int k = 0; k < 3; k++)
    check_hip(hipMemcpyAsync(G->model + k * G->ne, m[k], G->ne * sizeof(double), hipMemcpyHostToDevice, mp->stream),
              "model H2D");
  check_hip(hipMemcpyAsync(G->jac, jacobian, G->ne * sizeof(float), hipMemcpyHostToDevice, mp->stream), "model H2D");
  check_hip(hipStreamSynchronize(mp->stream), "sf2d_grad_set_model");
}
int sf2d_grad_has_model(long* Mesh_pointer) {
  const GradState* G = need(handle(Mesh_pointer));
  return G->model != nullptr || !G->h_model.empty();
}

// d chi / d (rho, vp, vs) [3][nspec][25] in ispec order and (parts not null) d chi / d (kappa, mu, rho through the mass,
// rho vp, rho vs) [5][nspec][25].  Formed in the segment's state slots, which the sweep no longer needs, as many elements at
// a time as they hold (all of them where a segment has at least seven steps).
void sf2d_grad_model_result(long* Mesh_pointer, float dto2, double* grad, double* parts) {
  Mesh* mp = handle(Mesh_pointer);
  GradState* G = need(mp);
  const bool resident = G->model != nullptr;
  if (!resident && G->h_model.empty()) fail("sf2d_grad_model_result: call sf2d_grad_set_model first");
  const int nout = parts ? 8 : 3;
  const std::vector<int4> where = accumulator_places(mp, G);
  // the scratch memory: ispec_of_pos, then of the elements in hand where, (model, Jacobian) and the result
  const size_t per = sizeof(int4) + NGLL2 * (nout * sizeof(double) + (resident ? 0 : 3 * sizeof(double) + sizeof(float)));
  const size_t order_bytes = G->nf ? ((size_t)mp->nspec * sizeof(int) + 15) / 16 * 16 : 0;
  size_t room = 3 * G->nfield * G->chunk * sizeof(float);
  char* base = reinterpret_cast<char*>(G->seg);
  char* own = nullptr;
  const size_t few = order_bytes + per * std::min(mp->nspec, 64);
  if (room < few) base = own = device_alloc<char>(room = few);  // meshes of a few elements, segments of one step
  const int most = (int)std::min<size_t>(mp->nspec, (room - order_bytes) / per);
  auto put = [&](void* dst, const void* src, size_t bytes) {
    check_hip(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, mp->stream), "gradient H2D");
  };
  int* const order = reinterpret_cast<int*>(base);
  if (G->nf) put(order, mp->ispec_of_pos.data(), (size_t)mp->nspec * sizeof(int));
  for (int e0 = 0; e0 < mp->nspec; e0 += most) {
    const int n = std::min(most, mp->nspec - e0);
    const size_t np = (size_t)n * NGLL2, l0 = element_point(e0);
    int4* const at = reinterpret_cast<int4*>(base + order_bytes);
    double* const out = reinterpret_cast<double*>(at + n);
    put(at, where.data() + e0, n * sizeof(int4));
    const double* model = G->model + l0;
    const float* jac = G->jac + l0;
    if (!resident) {
      double* const m = out + nout * np;
      for (int k = 0; k < 3; k++) put(m + k * np, G->h_model.data() + k * G->ne + l0, np * sizeof(double));
      put(m + 3 * np, G->h_jac.data() + l0, np * sizeof(float));
      model = m;
      jac = reinterpret_cast<const float*>(m + 3 * np);
    }
    const long mstride = (long)(resident ? G->ne : np);
    hipLaunchKernelGGL(k_grad_model, dim3((unsigned)((np + GT - 1) / GT)), dim3(GT), 0, mp->stream, (long)np, mstride, at,
                       mp->d_ibool, G->gk, G->gm, G->pm, model, jac, out, parts ? 1 : 0, mp->basis);
    check_hip(hipGetLastError(), "k_grad_model launch");
    if (G->nf) {
      hipLaunchKernelGGL(k_grad_model_stacey, dim3((unsigned)((G->nf + 63) / 64)), dim3(64), 0, mp->stream, stacey_faces(mp),
                         e0, (long)np, mstride, order, G->gvp, G->gvs, G->pm, model, (double)dto2, out, parts ? 1 : 0);
      check_hip(hipGetLastError(), "k_grad_model_stacey launch");
    }
    auto get = [&](double* dst, int c0, int nc) {  // components c0 .. c0 + nc - 1 of the range
      for (int c = 0; c < nc; c += n == mp->nspec ? nc : 1)
        check_hip(hipMemcpyAsync(dst + c * G->ne + l0, out + (c0 + c) * np, (n == mp->nspec ? nc : 1) * np * sizeof(double),
                                 hipMemcpyDeviceToHost, mp->stream),
                  "gradient D2H");
    };
    get(grad, 0, 3);
    if (parts) get(parts, 3, 5);
  }
  check_hip(hipStreamSynchronize(mp->stream), "sf2d_grad_model_result");
  device_free(own);
}

// replaces the materials of a prepared handle: kappa, mu, rho vp, rho vs [nspec][25] in ispec order and the
// inverse mass rmassx, rmassz [nglob] in the caller's numbering
void sf2d_mesh_set_materials(long* Mesh_pointer, const float* kappav, const float* muv, const float* rho_vp,
                             const float* rho_vs, const float* rmassx, const float* rmassz) {
  Mesh* mp = handle(Mesh_pointer);
  if (!mp->sorted) fail("sf2d_mesh_set_materials: prepare_fields_elastic_device was not called");
  flush_correctors(mp);
  check_hip(hipStreamSynchronize(mp->stream), "sf2d_mesh_set_materials");
  const size_t ne = (size_t)mp->nspec * NGLL2;
  auto put = [&](float* dev, const float* host) {
    if (!dev || !host) return;
    std::vector<float> v = to_device_order(mp, host);
    check_hip(hipMemcpy(dev, v.data(), ne * sizeof(float), hipMemcpyHostToDevice), "materials H2D");
  };
  put(mp->d_kappav, kappav);
  put(mp->d_muv, muv);
  if (mp->d_moduli && (kappav || muv)) {
    launch_pack_elements(mp);
    check_hip(hipStreamSynchronize(mp->stream), "pack elements");
  }
  put(mp->d_rho_vp, rho_vp);
  put(mp->d_rho_vs, rho_vs);
  if (rmassx) points_to_device(mp, mp->d_rmassx, rmassx, 1, "rmassx H2D");
  if (rmassz) points_to_device(mp, mp->d_rmassz, rmassz, 1, "rmassz H2D");
  if (mp->tower && (rmassx || rmassz) && !(rmassx && rmassz && tower_masses_fit(mp, rmassx, rmassz))) tower_release(mp);
  if (rmassx || rmassz) mp->same_mass = 0;  // the Newmark kernels read both arrays from here on
}

}  // extern "C"
