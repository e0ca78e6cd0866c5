// A whole time step of the solid in two launches: towers of chains, then the points between them.
//
// A tower is a stack of chains (rows of up to 12 elements) in which each chain's top GLL row is the next one's bottom
// row.  One wave walks up a tower, lane 5 k + i holding column i of element k, and carries the displacement and the
// force of the shared GLL row in registers from one chain to the next.  A GLL point inside a tower gets all of its
// force there, so the wave applies the Newmark corrector of this step and the predictor of the next one to it at once
// and in place: nobody else reads or writes the point.  Per step such a point costs its displacement and velocity read
// and written, its inverse mass, and the element data once: no acceleration array, no second pass, no colours.
//
// The other points -- the tower's outline and every point that something else also acts on or looks at (absorbing
// edges, sources, fluid-solid edges, CPML elements, receivers, points whose two inverse masses differ) -- are the
// interface.  For these the wave stores its force into a slot of its own, further workgroups of the same launch add the
// boundary terms into accel, and the interface kernel sums the boundary terms and the slots of each point in the order in
// which a launch per colour adds them, clears accel and makes the same Newmark update.
//
// State between two such steps: (d_n, v'_n) predicted, accel zero at the interface points with a boundary term and
// stale elsewhere.  A run starts from the ordinary predictor; its last step leaves displacement, velocity and
// acceleration as the callers know them.
//
// What bounds it: on large meshes HBM.  2000 x 1000 elements (32 M points): k_tower moves 1.74 GB in 371 us (4.7 TB/s, what a
// copy reaches on this card), k_interface 0.17 GB in 31 us; four colour launches and a corrector-predictor pass took 576 us.
// On small meshes the latency of launches and dependent loads: 80 x 60 elements 6.0 and 3.2 us.
#include <algorithm>
#include <cstdlib>
#include <vector>

#include "sf2d_mesh.h"
#include "sf2d_tower.h"
#include "specfem2d_gpu_ext.h"

namespace sf2d {

struct TowerState {
  TowerPlan plan;
  float2* d_layer = nullptr; // forces of the CPML layer's element points
  // adjoint runs and SAVE_FORWARD runs: `store_steps` steps of Stacey terms [face point] (those from step store_first on);
  // the second displacement arrays and the boundary terms of the two fields of an adjoint run [nglob]
  float2* d_store = nullptr;
  int store_steps = 0, store_first = -1;
  float* d_other[2] = {nullptr, nullptr};
  float2* d_acc[2] = {nullptr, nullptr};
  float2* d_slot = nullptr;  // [slot_shots][plan.nslot] forces of interface points
  int slot_shots = 0;
  int geo = 0;               // k_tower's GEO
};

namespace {

constexpr int TROW = 64;  // float2 per GLL row in LDS, in lane order: writes and reads without bank conflicts

// attenuation state and coefficient sets in the chain kernel's lane order (att_load); SETS: 0 no attenuation, 1 one
// coefficient set for every point, 2 a set index per point
struct TowerAtt {
  const unsigned int* idx;
  const float4* table;
  float* state;
  long ne;
};

template <typename T>
__device__ __forceinline__ void st_off(T* base, unsigned byte_off, T value) {
  *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + byte_off) = value;
}

// The wavefields of a step, shot s at s * stride points: (d, v) = (d_n, v'_n) in, (d_out, v_out) = (d_{n+1}, v'_{n+1})
// out, which may be the same arrays.  r_out (may be null): the force r_n of every point.  last 1: the step ends a run
// instead, accel = a_n and v_out = v_n; 2: r_out only.  accel holds the boundary terms at interface points.
struct TowerFields {
  const float2 *d, *v;
  float2 *d_out, *v_out, *r_out, *accel;
  long stride;
  int nshot, last;
  struct Row {  // a point's operands besides the field that the force is computed from
    float2 v;
  };
  __device__ long ref(int shot) const { return shot * stride; }
  __device__ const float2* field(long shot) const { return d + shot; }
  __device__ Row load(long shot, unsigned o) const { return {ld_off(v + shot, o)}; }
  // the point at byte offset o: corrector of this step and predictor of the next (k_corrector's and k_predictor's
  // operations, contracted the same way, so that a run in pieces gives the bits of the run in one) from the force r
  __device__ void update(const Newmark& c, long shot, unsigned o, float2 r, float wx, float wz, float2 d, Row q) const {
    if (r_out) st_off(r_out + shot, o, r);
    if (last == 2) return;
    float2 v = q.v;
    const float2 a = make_float2(r.x * wx, r.y * wz);
    v.x = fmaf(c.dto2, a.x, v.x);
    v.y = fmaf(c.dto2, a.y, v.y);
    if (last) {
      st_off(accel + shot, o, a);
    } else {
      d.x = fmaf(c.dt2o2, a.x, fmaf(c.dt, v.x, d.x));
      d.y = fmaf(c.dt2o2, a.y, fmaf(c.dt, v.y, d.y));
      v.x = fmaf(c.dto2, a.x, v.x);
      v.y = fmaf(c.dto2, a.y, v.y);
      st_off(d_out + shot, o, d);
    }
    st_off(v_out + shot, o, v);
  }
};

// The fields of a reverse step (gradient.hip): R~_n in, from which the force is computed, the cotangents D and V', and
// R~_{n-1} = W A out: D += -K R~; V = V' + dt D; A = dt/2 V' + dt^2/2 D + dt/2 V
struct AdjointFields {
  const float2* Rb;
  float2 *Rb_out, *D, *Vb;  // Rb_out may be Rb
  long stride;
  int nshot;
  struct Row {
    float2 D, Vb;
  };
  __device__ long ref(int shot) const { return shot * stride; }
  __device__ const float2* field(long shot) const { return Rb + shot; }
  __device__ Row load(long shot, unsigned o) const { return {ld_off(D + shot, o), ld_off(Vb + shot, o)}; }
  __device__ void update(const Newmark& c, long shot, unsigned o, float2 r, float wx, float wz, float2, Row q) const {
    float2 db = q.D, v, a;
    db.x += r.x;
    db.y += r.y;
    v.x = q.Vb.x + c.dt * db.x;
    v.y = q.Vb.y + c.dt * db.y;
    a.x = c.dto2 * q.Vb.x + c.dt2o2 * db.x;
    a.y = c.dto2 * q.Vb.y + c.dt2o2 * db.y;
    a.x = a.x + c.dto2 * v.x;
    a.y = a.y + c.dto2 * v.y;
    st_off(D + shot, o, db);
    st_off(Vb + shot, o, v);
    st_off(Rb_out + shot, o, make_float2(wx * a.x, wz * a.y));
  }
};

// The two fields of an adjoint run (SIMULATION_TYPE 3) as two shots: 0 the adjoint field, 1 the reconstructed one, which
// steps backwards.  As TowerFields, with the outputs in other arrays than the inputs: the kernels need the step's two
// displacements and the adjoint acceleration (a0).  last: the step ends the run, a0 and a1 = a_n, (v0_out, v1_out) = v_n.
struct PairFields {
  const float2 *d0, *v0, *d1, *v1;
  float2 *d0_out, *v0_out, *a0, *d1_out, *v1_out, *a1;
  float2 *acc0, *acc1;       // boundary terms, zero between the steps
  Newmark nm0, nm1;
  int nshot, last;
  struct Row {
    float2 v;
  };
  __device__ int ref(int shot) const { return shot; }
  __device__ const float2* field(int s) const { return s ? d1 : d0; }
  __device__ Row load(int s, unsigned o) const { return {ld_off(s ? v1 : v0, o)}; }
  __device__ void update(const Newmark&, int s, unsigned o, float2 r, float wx, float wz, float2 d, Row q) const {
    const float dto2 = s ? nm1.dto2 : nm0.dto2, dt = s ? nm1.dt : nm0.dt, dt2o2 = s ? nm1.dt2o2 : nm0.dt2o2;
    const float2 a = make_float2(r.x * wx, r.y * wz);
    float2 v = q.v;
    v.x = fmaf(dto2, a.x, v.x);
    v.y = fmaf(dto2, a.y, v.y);
    if (s == 0 || last) st_off(s ? a1 : a0, o, a);
    if (!last) {
      d.x = fmaf(dt2o2, a.x, fmaf(dt, v.x, d.x));
      d.y = fmaf(dt2o2, a.y, fmaf(dt, v.y, d.y));
      v.x = fmaf(dto2, a.x, v.x);
      v.y = fmaf(dto2, a.y, v.y);
      st_off(s ? d1_out : d0_out, o, d);
    }
    st_off(s ? v1_out : v0_out, o, v);
  }
};

// What else the launch does, in workgroups after the towers': Stacey faces, sources, receivers and fluid-solid edges of
// the step
struct TowerEdges {
  StaceyFaces faces;
  SourceSet sources;
  ReceiverSet receivers;
  int it;                  // 0-based time sample
  int nface_wg, nsource, nreceiver, ncoupling_wg;
  CouplingPoints coupling; // fluid-solid edges (one shot)
  const float* pdd;        // the fluid's acceleration there
  const int* step;         // (may be null) the 1-based step in device memory in place of it
  const int* src_shot;     // shot of each source (null: one shot)
  float* seismo;           // [shot][2][receiver][time]
  long seismo_stride;
  float2* store;           // SAVE_FORWARD: the Stacey terms of the step, [face point] (one shot; null: not kept)
  int wgs(int nshot) const { return nface_wg * nshot + nsource + nreceiver * nshot + ncoupling_wg; }
};

__device__ __forceinline__ void tower_edges(const TowerEdges& E, const TowerFields& F, int wg) {
  const int faces = E.nface_wg * F.nshot;
  const int it = E.step ? *E.step - 1 : E.it;
  if (wg < faces) {
    const int shot = wg / E.nface_wg;
    const int q = (wg - shot * E.nface_wg) * 64 + threadIdx.x;
    const float2 f = stacey_traction(E.faces, q, F.v + shot * F.stride, (float*)(F.accel + shot * F.stride), 1);
    if (E.store && q < E.faces.nabs * NGLL) E.store[q] = f;
    return;
  }
  wg -= faces;
  if (wg < E.nsource) {
    const long shot = E.src_shot ? E.src_shot[wg] : 0;
    source_force(E.sources, wg, threadIdx.x, it, (float*)(F.accel + shot * F.stride), 1);
    return;
  }
  wg -= E.nsource;
  if (wg >= E.nreceiver * F.nshot) {
    couple_solid(E.coupling, (wg - E.nreceiver * F.nshot) * 64 + threadIdx.x, E.pdd, 1.f, (float*)F.accel);
    return;
  }
  const int shot = wg / E.nreceiver, r = wg - shot * E.nreceiver;
  if (E.faces.is_elastic[E.receivers.ispec[r]])  // receivers in fluid elements are recorded by the fluid
    record_receiver(E.receivers, r, threadIdx.x, it, F.d + shot * F.stride, E.seismo + shot * E.seismo_stride, 1);
}

// the boundary part of a reverse step: residuals into D, -B R~ into V', and the Stacey terms of the gradient
struct AdjointEdges {
  StaceyFaces faces;
  ReceiverSet receivers;
  int nface_wg, nreceiver;
  const float* res;        // [shot][receiver][2] of the step
  const float2* vpn;       // v'_n of the forward field
  float *gvp, *gvs;
  int wgs(int nshot) const { return nface_wg * (nshot + 1) + nreceiver * nshot; }
};

__device__ __forceinline__ void tower_edges(const AdjointEdges& E, const AdjointFields& F, int wg) {
  if (wg < E.nface_wg) {
    stacey_gradient(E.faces, wg * 64 + threadIdx.x, F.nshot, 1, F.stride, E.vpn, F.Rb, E.gvp, E.gvs);
    return;
  }
  wg -= E.nface_wg;
  const int faces = E.nface_wg * F.nshot;
  if (wg < faces) {
    const int shot = wg / E.nface_wg;
    stacey_traction(E.faces, (wg - shot * E.nface_wg) * 64 + threadIdx.x, F.Rb + shot * F.stride,
                    (float*)(F.Vb + shot * F.stride), 1);
    return;
  }
  wg -= faces;
  const int shot = wg / E.nreceiver, r = wg - shot * E.nreceiver;
  adjoint_receiver(E.receivers, r, threadIdx.x, E.res + (size_t)shot * 2 * E.receivers.nrec,
                   (float*)(F.D + shot * F.stride), 1);
}

// the boundary part of a step of an adjoint run: Stacey edges, adjoint sources and receivers of the adjoint field, the
// forward run's stored Stacey terms and its sources for the reconstructed one
struct PairEdges {
  StaceyFaces faces;
  ReceiverSet receivers;
  SourceSet sources;
  int it, cur, nstep;      // 0-based samples of the forward run's time and of the seismograms
  int nface_wg, nsource, nadj, nreceiver;
  const float* adj;        // [2][nstep][receiver]
  const float2* store;     // [face point]
  float* seismo;
  int wgs(int) const { return 2 * nface_wg + nsource + nadj + nreceiver; }
};

__device__ __forceinline__ void tower_edges(const PairEdges& E, const PairFields& F, int wg) {
  const int t = threadIdx.x;
  if (wg < E.nface_wg) {
    stacey_traction(E.faces, wg * 64 + t, F.v0, (float*)F.acc0, 1);
    return;
  }
  wg -= E.nface_wg;
  if (wg < E.nface_wg) {
    stored_traction(E.faces, wg * 64 + t, E.store, (float*)F.acc1);
    return;
  }
  wg -= E.nface_wg;
  if (wg < E.nsource) {
    source_force(E.sources, wg, t, E.it, (float*)F.acc1, 1);
    return;
  }
  wg -= E.nsource;
  if (wg < E.nadj) {
    adjoint_source(E.receivers, E.faces.is_elastic, wg, t, E.it, E.nstep, E.adj, (float*)F.acc0);
    return;
  }
  record_receiver(E.receivers, wg - E.nadj, t, E.cur, F.d0, E.seismo, 1);
}

// The operands of a lane's column of one chain that the next iteration starts from, loaded one chain ahead: the
// displacement of GLL rows 1 .. 4, the moduli of rows 0 .. 4, the element's geometry record
struct ChainRegs {
  float2 d[NGLL - 1], mod[NGLL];
  float4 ge;
};

// GEO: 0 every element a rectangle {xi_x, gamma_z}, 1 every element affine (one record), 2 geometry per point; 3 and 4 are 1
// and 2 with offsets that count from the tower's first element, for element arrays that pass 4 GiB (tower_geometry: a base
// of the tower's own costs scalar registers that the kernel has too few of already, 1 to 2.5 percent of a small mesh's step)
template <int GEO, int SETS, class Fields, class Edges>
__global__ __launch_bounds__(64) void k_tower(
    int ntower, const int4* __restrict__ desc, const int4* __restrict__ rows, const float4* __restrict__ geom,
    const float4* __restrict__ geom_elem, const float2* __restrict__ mod, const Fields F,
    const float* __restrict__ rm, float2* __restrict__ slot, int nslot, const Newmark nm, const Basis basis,
    const TowerAtt att, int tower_wgs, const Edges edges) {
  constexpr bool RECT = GEO == 0, WIDE = GEO >= 3, PER_POINT = GEO == 2 || GEO == 4;
  __shared__ float2 s_t[NGLL * TROW + 1];
  if ((int)blockIdx.x >= tower_wgs) {
    tower_edges(edges, F, blockIdx.x - tower_wgs);
    return;
  }
  // the shots of a tower are neighbours on one XCD: its element data comes from HBM once
  const int item = (blockIdx.x % NXCD) * (tower_wgs / NXCD) + blockIdx.x / NXCD;
  const int tower = F.nshot == 1 ? item : item / F.nshot;
  if (tower >= ntower) return;  // uniform over the wave
  const int shot = item - tower * F.nshot;
  const auto at = F.ref(shot);
  const float2* const __restrict__ d = F.field(at);
  slot += (size_t)shot * nslot;
  const int4 td = desc[4 * tower], tb = desc[4 * tower + 1], ts = desc[4 * tower + 2], tt = desc[4 * tower + 3];
  const int nch = td.y, ne = td.z;
  const int4* const row = rows + td.w;
  const int lane = threadIdx.x;
  const int k = min(lane / NGLL, Mesh::CHAIN_ELEMS);
  const int i = lane % NGLL;
  const int kk = min(k, ne - 1);
  const int x = 4 * kk + i;
  const int xe = 4 * ne;
  const bool active = lane / NGLL < ne;
  const bool writer = active && (i < NGLL - 1 || k == ne - 1);
  const unsigned below_lo = x < 32 ? (1u << x) - 1u : ~0u, below_hi = x < 32 ? 0u : (1u << (x - 32)) - 1u;
  float hpi[NGLL], hwi[NGLL];  // this lane's row of the derivative matrix and column of the weighted one
#pragma unroll
  for (int m = 0; m < NGLL; m++) {
    hpi[m] = basis.hp[i * NGLL + m];
    hwi[m] = basis.hpw[m * NGLL + i];
  }
  const float wi = basis.w[i];
  // byte offsets of this lane's points (fields of 8 bytes): in row 0 of the current chain, in its row 1 (from there the
  // rows go up by `up`), in the tower's topmost row; and its word of row 0 of the chain in the element arrays
  auto point = [&](const int4 r) { return 8u * (unsigned)(x == 0 ? r.y : x == xe ? r.z : r.x + x); };
  unsigned off0 = point(tb), off1 = point(ts);
  const unsigned offt = point(tt);
  const unsigned up = 8u * (x == 0 || x == xe ? 1u : (unsigned)(xe - 1));
  const unsigned first = WIDE ? 0u : (unsigned)td.x;
  const unsigned att0 = WIDE ? (unsigned)td.x * NGLL2 : 0u;  // indices, not bytes: within 32 bits
  unsigned word = first * NGLL2 + (unsigned)min(lane, NGLL * ne - 1);
  unsigned elem = first + (unsigned)kk;
  if (WIDE) {
    mod = at_element(mod, td.x);
    geom = at_element(geom, td.x);
    geom_elem += td.x;
  }
  const unsigned mrow = (unsigned)(NGLL * ne);

  auto load_chain = [&](unsigned o1, bool top, unsigned w, unsigned e, ChainRegs& q) {
#pragma unroll
    for (int j = 0; j < NGLL - 2; j++) q.d[j] = ld_off(d, o1 + (unsigned)j * up);
    q.d[NGLL - 2] = ld_off(d, top ? offt : o1 + (unsigned)(NGLL - 2) * up);
#pragma unroll
    for (int j = 0; j < NGLL; j++) q.mod[j] = ld_off(mod, 8u * (w + (unsigned)j * mrow));
    if (!PER_POINT) q.ge = ld_off(geom_elem, 16u * e);
  };
  // the update of one row's point, or its share of an interface point
  auto finish = [&](const int4 r, unsigned o, float2 f, float2 u, const typename Fields::Row& vp, float m) {
    if (!writer) return;
    const unsigned bits = x < 32 ? (unsigned)r.x >> x : (unsigned)r.y >> (x - 32);
    if (bits & 1u) {
      slot[r.z + __popc((unsigned)r.x & below_lo) + __popc((unsigned)r.y & below_hi)] = f;
    } else {
      F.update(nm, at, o, f, m, m, u, vp);
    }
  };

  auto edge_bit = [&](const int4 r) { return ((xe < 32 ? (unsigned)r.x >> xe : (unsigned)r.y >> (xe - 32)) & 1u) != 0; };
  float2 u0 = ld_off(d, off0);
  float2 carry = make_float2(0.f, 0.f);
  ChainRegs nx;
  load_chain(off1, nch == 1, word, elem, nx);
  float4 cf[3];
  if (SETS == 1) {
#pragma unroll
    for (int s = 0; s < 3; s++) cf[s] = att.table[s];
  }
  const float2* const el = s_t + NGLL * k;  // this element's five points of GLL row 0

  for (int c = 0; c < nch; c++) {
    const ChainRegs q = nx;
    // this chain's velocity and inverse mass (rows 0 .. 3), needed at its end
    typename Fields::Row vp[NGLL - 1];
    float ms[NGLL - 1];
#pragma unroll
    for (int j = 0; j < NGLL - 1; j++) {
      const unsigned o = j == 0 ? off0 : off1 + (unsigned)(j - 1) * up;
      vp[j] = F.load(at, o);
      ms[j] = ld_off(rm, o / 2u);
    }
    float4 st[3];  // attenuation state of the next row
    if (SETS > 0) {
#pragma unroll
      for (int s = 0; s < 3; s++) st[s] = reinterpret_cast<const float4*>(att.state)[(size_t)s * att.ne + (att0 + word)];
    }
    const unsigned noff = off1 + 4u * up, nword = word + (unsigned)NGLL * mrow, nelem = elem + (unsigned)ne;
    if (c + 1 < nch) load_chain(noff, c + 2 == nch, nword, nelem, nx);
    float2 u[NGLL];
    u[0] = u0;
#pragma unroll
    for (int j = 1; j < NGLL; j++) u[j] = q.d[j - 1];

    // xi derivatives: the element's rows through LDS
#pragma unroll
    for (int j = 0; j < NGLL; j++) s_t[j * TROW + lane] = u[j];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float2 t1[NGLL], t2[NGLL];
#pragma unroll
    for (int j = 0; j < NGLL; j++) {
      float dux_dxi = 0.f, duz_dxi = 0.f;
#pragma unroll
      for (int m = 0; m < NGLL; m++) {
        const float2 e = el[j * TROW + m];
        dux_dxi += e.x * hpi[m];
        duz_dxi += e.y * hpi[m];
      }
      float dux_dga = 0.f, duz_dga = 0.f;
#pragma unroll
      for (int m = 0; m < NGLL; m++) {
        const float h = basis.hp[j * NGLL + m];
        dux_dga += u[m].x * h;
        duz_dga += u[m].y * h;
      }
      const float kap = q.mod[j].x, mu = q.mod[j].y;
      const float lambdal = kap - mu, lp2m = kap + mu;
      float4 gp = q.ge;
      if (PER_POINT) gp = ld_off(geom, 16u * (elem * NGLL2 + (unsigned)(j * NGLL + i)));
      const float xixl = gp.x, xizl = RECT ? 0.f : gp.y, gaxl = RECT ? 0.f : gp.z, gazl = gp.w;
      const float dux_dxl = RECT ? dux_dxi * xixl : dux_dxi * xixl + dux_dga * gaxl;
      const float dux_dzl = RECT ? dux_dga * gazl : dux_dxi * xizl + dux_dga * gazl;
      const float duz_dxl = RECT ? duz_dxi * xixl : duz_dxi * xixl + duz_dga * gaxl;
      const float duz_dzl = RECT ? duz_dga * gazl : duz_dxi * xizl + duz_dga * gazl;
      // contracted as in k_elastic_forces_col, so that both kernels give the same bits
      float sxx = fmaf(lp2m, dux_dxl, lambdal * duz_dzl);
      float szz = fmaf(lambdal, dux_dxl, lp2m * duz_dzl);
      float sxz = mu * (RECT && SETS == 0 ? fmaf(duz_dxi, xixl, dux_dzl) : duz_dxl + dux_dzl);
      if (SETS > 0) {
        const unsigned la = att0 + word + (unsigned)j * mrow;
        float ev[9] = {st[0].x, st[0].y, st[0].z, st[0].w, st[1].x, st[1].y, st[1].z, st[1].w, st[2].x};
        float ov[3] = {st[2].y, st[2].z, st[2].w};
        if (j + 1 < NGLL) {
#pragma unroll
          for (int s = 0; s < 3; s++)
            st[s] = reinterpret_cast<const float4*>(att.state)[(size_t)s * att.ne + la + mrow];
        }
        if (SETS == 2) {
          const float4* coef = att.table + 3 * (size_t)att.idx[la];
#pragma unroll
          for (int s = 0; s < 3; s++) cf[s] = coef[s];
        }
        attenuate_point(cf, ev, ov, kap, mu, dux_dxl, dux_dzl, duz_dxl, duz_dzl, sxx, sxz, szz);
        if (active) att_store(att.state, att.ne, la, ev, ov);
      }
      if (RECT) {  // xi_z = gamma_x = 0: J xi_x = 1 / gamma_z, J gamma_z = 1 / xi_x
        const float cx = 1.f / gazl, cz = 1.f / xixl;
        t1[j] = make_float2(cx * sxx, cx * sxz);
        t2[j] = make_float2(cz * sxz, cz * szz);
      } else {
        const float jac = 1.f / (xixl * gazl - gaxl * xizl);
        t1[j] = make_float2(jac * fmaf(xixl, sxx, xizl * sxz), jac * fmaf(xixl, sxz, xizl * szz));
        t2[j] = make_float2(jac * fmaf(gaxl, sxx, gazl * sxz), jac * fmaf(gaxl, sxz, gazl * szz));
      }
    }
    // xi flux contraction: the element's rows through LDS
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < NGLL; j++) s_t[j * TROW + lane] = t1[j];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float2 f[NGLL];
#pragma unroll
    for (int j = 0; j < NGLL; j++) {
      float sx = 0.f, sz = 0.f;
#pragma unroll
      for (int m = 0; m < NGLL; m++) {
        const float2 e = el[j * TROW + m];
        sx += e.x * hwi[m];
        sz += e.y * hwi[m];
      }
      float gx = 0.f, gz = 0.f;
#pragma unroll
      for (int m = 0; m < NGLL; m++) {
        const float h = basis.hpw[m * NGLL + j];
        gx += t2[m].x * h;
        gz += t2[m].y * h;
      }
      const float wj = basis.w[j];
      f[j] = make_float2(-(wj * sx + wi * gx), -(wj * sz + wi * gz));
    }
    __builtin_amdgcn_wave_barrier();
    // the shared column's force moves from element k - 1 (lane 5 k - 1) to element k (lane 5 k)
#pragma unroll
    for (int j = 0; j < NGLL; j++) {
      const float fx = __shfl_up(f[j].x, 1, 64);
      const float fz = __shfl_up(f[j].y, 1, 64);
      if (i == 0 && k > 0) {
        f[j].x += fx;
        f[j].y += fz;
      }
    }
    // the row below's force, or where the columns are interface points a slot of its own
    const int4 r0 = row[4 * c];
    const bool lone = writer && c > 0 && ((x == 0 && (r0.x & 1)) || (x == xe && edge_bit(r0)));
    if (lone) {
      slot[r0.w + (x == 0 ? 0 : r0.x & 1)] = carry;
    } else {
      f[0].x += carry.x;
      f[0].y += carry.y;
    }
#pragma unroll
    for (int j = 0; j < NGLL - 1; j++) finish(j == 0 ? r0 : row[4 * c + j], j == 0 ? off0 : off1 + (unsigned)(j - 1) * up, f[j], u[j], vp[j], ms[j]);
    carry = f[NGLL - 1];
    u0 = u[NGLL - 1];
    off0 = off1 + (unsigned)(NGLL - 2) * up;
    off1 = noff;
    word = nword;
    elem = nelem;
  }
  // the tower's top row
  finish(row[4 * nch], offt, carry, u0, F.load(at, offt), ld_off(rm, offt / 2u));
}

// Interface points: the slots of each point summed in order, the boundary terms of accel added and cleared, and the
// Newmark update; old (CPML layer points): u + dt^2 / 4 a of this step, the layer's previous-step field, zero on the
// layer's outer boundary, whose displacement and velocity are zero when the next step starts (pml_boundary_elastic;
// IF_KEEP: not before the fluid has read them).
__global__ __launch_bounds__(IF_T) void k_interface(const InterfaceArgs A, const float2* __restrict__ slot, int nslot,
                                                   const TowerFields F, const float* __restrict__ rmx,
                                                   const float* __restrict__ rmz, const Newmark nm,
                                                   const float2* __restrict__ layer, float2* __restrict__ old,
                                                   float dt2o4) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= A.n) return;
  const long at = blockIdx.y * F.stride;
  const int g = A.id[q];
  const int fl = A.flag[q];
  const SlotIds s = slot_ids(A, q);
  const float2 dd = F.d[at + g], vv = F.v[at + g];
  const float wx = rmx[g], wz = rmz[g];
  float2 acc = make_float2(0.f, 0.f);
  if (fl & IF_ACC) acc = F.accel[at + g];
  const SlotValues<float2> x = slot_values(q >= A.n2, s.t, slot + (size_t)blockIdx.y * nslot);
  SlotValues<float2> y{};
  if (q >= A.n4) y = slot_values(true, s.p, layer);
  const float2 r = sum_slots(s.p, y, sum_slots(s.t, x, acc));
  if ((fl & IF_ACC) && F.last != 1) F.accel[at + g] = make_float2(0.f, 0.f);
  if ((fl & IF_PML) && old) {
    const float ax = r.x * wx, az = r.y * wz;
    old[g] = (fl & IF_PML_EDGE) ? make_float2(0.f, 0.f)
                                : make_float2(fmaf(dt2o4, ax, dd.x), fmaf(dt2o4, az, dd.y));
  }
  if ((fl & (IF_PML_EDGE | IF_KEEP)) == IF_PML_EDGE && !F.last) {
    F.d_out[at + g] = make_float2(0.f, 0.f);
    F.v_out[at + g] = make_float2(0.f, 0.f);
    return;
  }
  F.update(nm, at, 8u * (unsigned)g, r, wx, wz, dd, {vv});
}

__global__ __launch_bounds__(IF_T) void k_interface_adjoint(const InterfaceArgs A, const float2* __restrict__ slot,
                                                           int nslot, const AdjointFields F,
                                                           const float* __restrict__ rmx, const float* __restrict__ rmz,
                                                           const Newmark nm) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= A.n) return;
  const long at = blockIdx.y * F.stride;
  const int g = A.id[q];
  const SlotIds s = slot_ids(A, q);
  const AdjointFields::Row row = F.load(at, 8u * (unsigned)g);
  const float wx = rmx[g], wz = rmz[g];
  const SlotValues<float2> x = slot_values(q >= A.n2, s.t, slot + (size_t)blockIdx.y * nslot);
  const float2 r = sum_slots(s.t, x, make_float2(0.f, 0.f));
  F.update(nm, at, 8u * (unsigned)g, r, wx, wz, make_float2(0.f, 0.f), row);
}

__global__ __launch_bounds__(IF_T) void k_interface_pair(const InterfaceArgs A, const float2* __restrict__ slot, int nslot,
                                                        const PairFields F, const float* __restrict__ rmx,
                                                        const float* __restrict__ rmz) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= A.n) return;
  const int f = blockIdx.y;
  const int g = A.id[q];
  const int fl = A.flag[q];
  const SlotIds s = slot_ids(A, q);
  const float2 d = F.field(f)[g];
  const PairFields::Row row = F.load(f, 8u * (unsigned)g);
  const float wx = rmx[g], wz = rmz[g];
  float2 b = make_float2(0.f, 0.f);
  float2* const acc = f ? F.acc1 : F.acc0;
  if (fl & (IF_ACC | IF_LOOKED_AT)) b = acc[g];  // receivers' points take the adjoint sources
  const SlotValues<float2> x = slot_values(q >= A.n2, s.t, slot + (size_t)f * nslot);
  const float2 r = sum_slots(s.t, x, b);
  if (fl & (IF_ACC | IF_LOOKED_AT)) acc[g] = make_float2(0.f, 0.f);
  F.update(F.nm0, f, 8u * (unsigned)g, r, wx, wz, d, row);
}

// accel = 0 at the interface points with a boundary term (the start of a run of tower steps)
__global__ __launch_bounds__(256) void k_interface_clear(int n, const int* __restrict__ ids,
                                                         const uint8_t* __restrict__ flag, float2* __restrict__ accel,
                                                         long stride) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n && (flag[q] & IF_ACC)) accel[ids[q] + blockIdx.y * stride] = make_float2(0.f, 0.f);
}

// the slots of nshot fields; false (what is there stays) when the spare memory does not hold them
bool reserve_slots(Mesh* mp, int nshot) {
  TowerState* T = mp->tower;
  if (nshot <= T->slot_shots) return true;
  const size_t n = std::max<size_t>(1, (size_t)T->plan.nslot * nshot);
  if (n * sizeof(float2) > spare_memory()) return false;
  batch_drop_graph(mp);  // its launches hold the address
  device_free(T->d_slot);
  T->d_slot = device_alloc<float2>(n);
  T->slot_shots = nshot;
  return true;
}
float2* tower_slots(const TowerState* T, int nshot) {
  if (nshot > T->slot_shots) fail("fused step of %d fields: slots for %d", nshot, T->slot_shots);
  return T->d_slot;
}

// The kernel's GEO: offsets from the start of the element arrays where these stay below 4 GiB, 21.4 million elements of
// moduli and 10.7 of geometry per point (SF2D_WIDE_OFFSETS: from the tower on any mesh)
int tower_geometry(const Mesh* mp) {
  const bool affine = !mp->no_affine && mp->n_affine == mp->nspec;
  const size_t bytes = element_point(mp->nspec) * (affine ? sizeof(float2) : sizeof(float4));
  const bool wide = bytes >= ((size_t)1 << 32) || getenv("SF2D_WIDE_OFFSETS");
  if (affine) return wide ? 3 : mp->rect ? 0 : 1;
  return wide ? 4 : 2;
}

template <class Fields, class Edges, class Kernel>
void launch_k_tower(Mesh* mp, Kernel kern, const Fields& F, const Edges& E, float2* slot, const Newmark& nm) {
  const TowerPlan& P = mp->tower->plan;
  const TowerAtt att{mp->d_att_idx, mp->d_att_table, mp->d_att_e, (long)mp->nspec * NGLL2};
  const int wgs = (P.ntower * F.nshot + NXCD - 1) / NXCD * NXCD;
  hipLaunchKernelGGL(kern, dim3(wgs + E.wgs(F.nshot)), dim3(64), 0, mp->stream, P.ntower, P.d_desc, P.d_row, mp->d_geom,
                     mp->d_geom_elem, mp->d_col_mod, F, mp->d_rmassx, slot, P.nslot, nm, mp->basis, att, wgs, E);
  check_hip(hipGetLastError(), "k_tower launch");
}

// one step of the fields F at time step it (1-based): towers with the step's Stacey faces, sources, fluid-solid edges
// (forward) and (seismo not null) receivers, the CPML layer, the interface
void launch_tower(Mesh* mp, const TowerFields& F, int it, float* seismo, long seismo_stride, const int* src_shot,
                  const Newmark& nm, bool forward, const int* step = nullptr,
                  float2* store = nullptr) {
  const TowerPlan& P = mp->tower->plan;
  float2* const slot = tower_slots(mp->tower, F.nshot);
  TowerEdges E{};
  E.faces = stacey_faces(mp);
  E.sources = source_set(mp);
  E.receivers = receiver_set(mp);
  E.it = it - 1;
  E.nface_wg = mp->stacey ? (mp->num_abs * NGLL + 63) / 64 : 0;
  E.nsource = mp->nsources_local;
  E.nreceiver = seismo ? mp->nrec_local : 0;
  if (forward) E.coupling = acoustic_coupling(mp, &E.pdd);
  E.ncoupling_wg = (E.coupling.n + 63) / 64;
  E.src_shot = src_shot;
  E.seismo = seismo;
  E.seismo_stride = seismo_stride;
  E.store = store;
  E.step = step;
  const int sets = !mp->attenuation ? 0 : mp->att_ntable == 1 ? 1 : 2;
  using K = decltype(&k_tower<0, 0, TowerFields, TowerEdges>);
#define SF2D_SETS(g) {k_tower<g, 0, TowerFields, TowerEdges>, k_tower<g, 1, TowerFields, TowerEdges>, \
                      k_tower<g, 2, TowerFields, TowerEdges>}
  const K kern[5][3] = {SF2D_SETS(0), SF2D_SETS(1), SF2D_SETS(2), SF2D_SETS(3), SF2D_SETS(4)};
#undef SF2D_SETS
  launch_k_tower(mp, kern[mp->tower->geo][sets], F, E, slot, nm);
  if (forward) pml_elastic_slots(mp, mp->tower->d_layer);
  if (P.n == 0) return;
  hipLaunchKernelGGL(k_interface, dim3((P.n + IF_T - 1) / IF_T, F.nshot), dim3(IF_T), 0, mp->stream, interface_args(P), slot,
                     P.nslot, F, mp->d_rmassx, mp->d_rmassz, nm, mp->tower->d_layer,
                     F.last ? nullptr : (float2*)pml_old_field(mp, false), 0.5f * nm.dt2o2);
  check_hip(hipGetLastError(), "k_interface launch");
}

// accel = 0 at the interface points with a boundary term, before the first of a run of steps
void clear_interface(Mesh* mp, float2* accel, long stride, int nshot) {
  const TowerPlan& P = mp->tower->plan;
  if (P.n == 0) return;
  hipLaunchKernelGGL(k_interface_clear, dim3((P.n + 255) / 256, nshot), dim3(256), 0, mp->stream, P.n, P.d_id, P.d_flag,
                     accel, stride);
  check_hip(hipGetLastError(), "k_interface_clear launch");
}

}  // namespace

namespace {

// Stacey terms are kept on the device for as many steps as fit 64 MB and cross to or from the host together: a copy and a
// synchronisation per step cost more than a step of a small mesh (80 x 32 elements: 100 of 115 us).  Less where the spare
// memory is less than twice that; SF2D_STACEY_STEPS sets the steps.
size_t store_points(const Mesh* mp) { return (size_t)mp->num_abs * NGLL; }
void prepare_store(Mesh* mp, int nstep) {
  TowerState* T = mp->tower;
  const size_t step = store_points(mp) * sizeof(float2);
  if (step == 0 || T->d_store) return;
  size_t steps = std::min((size_t)64 << 20, spare_memory() / 2) / step;
  if (const char* env = getenv("SF2D_STACEY_STEPS")) steps = strtoull(env, nullptr, 10);
  T->store_steps = (int)std::max<size_t>(1, std::min<size_t>((size_t)nstep, steps));
  T->d_store = device_alloc<float2>(store_points(mp) * T->store_steps);
}

}  // namespace

bool tower_takes(Mesh* mp, int nshot) {
  const long per_shot = (mp->tower ? mp->tower->plan.ntower : 0) + (long)mp->num_abs * NGLL / 64 + 1 + mp->nrec_local;
  return mp->tower && per_shot * nshot + mp->nsources_local < (1L << 25) &&  // workgroups of 64: below 2^32 threads
         reserve_slots(mp, nshot);
}

// shot batches and gradients: nshot forward fields, shot s at s * stride points
void tower_begin_shots(Mesh* mp, float* accel, long stride, int nshot) {
  clear_interface(mp, (float2*)accel, stride, nshot);
}
void tower_step_shots(Mesh* mp, const ShotStep& S, int it, float deltat, float deltatsqover2, float deltatover2) {
  const TowerFields F{(const float2*)S.d, (const float2*)S.v, (float2*)S.d_out, (float2*)S.v_out, (float2*)S.r_out,
                      (float2*)S.accel, S.stride, S.nshot, S.last};
  launch_tower(mp, F, it, S.seismo, (long)2 * mp->nrec_local * mp->nstep, S.src_shot,
               {deltatover2, deltat, deltatsqover2}, false, S.step);
}
void tower_step_adjoint(Mesh* mp, const float* Rb, float* Rb_out, float* D, float* Vb, long stride, int nshot, const float* res,
                        const float* vpn, float* gvp, float* gvs, float dt, float h, float dto2) {
  const TowerPlan& P = mp->tower->plan;
  float2* const slot = tower_slots(mp->tower, nshot);
  const AdjointFields F{(const float2*)Rb, (float2*)Rb_out, (float2*)D, (float2*)Vb, stride, nshot};
  const Newmark nm{dto2, dt, h};
  AdjointEdges E{};
  E.faces = stacey_faces(mp);
  E.receivers = receiver_set(mp);
  E.nface_wg = mp->stacey ? (mp->num_abs * NGLL + 63) / 64 : 0;
  E.nreceiver = mp->nrec_local;
  E.res = res;
  E.vpn = (const float2*)vpn;
  E.gvp = gvp;
  E.gvs = gvs;
  using K = decltype(&k_tower<0, 0, AdjointFields, AdjointEdges>);
  const K kern[5] = {k_tower<0, 0, AdjointFields, AdjointEdges>, k_tower<1, 0, AdjointFields, AdjointEdges>,
                     k_tower<2, 0, AdjointFields, AdjointEdges>, k_tower<3, 0, AdjointFields, AdjointEdges>,
                     k_tower<4, 0, AdjointFields, AdjointEdges>};
  launch_k_tower(mp, kern[mp->tower->geo], F, E, slot, nm);
  if (P.n == 0) return;
  hipLaunchKernelGGL(k_interface_adjoint, dim3((P.n + IF_T - 1) / IF_T, nshot), dim3(IF_T), 0, mp->stream, interface_args(P),
                     slot, P.nslot, F, mp->d_rmassx, mp->d_rmassz, nm);
  check_hip(hipGetLastError(), "k_interface_adjoint launch");
}

// Chains per tower (nchain: times the shots): about one wave per slot of the card (4096 at four waves per SIMD) and at
// most 16.  A tall tower has few interface rows (1 in 4 x chains), a short one more waves in flight; a wave takes 2.3 us per
// chain.  Measured, ms of 300 steps of 600 x 300 elements (15,000 chains) at 1, 2, 4, 8, 16 chains: 12.9, 11.7, 10.7, 12.0,
// 17.2; 40 steps of 2000 x 1000 (167,000 chains) at 4, 8, 16: 17.1, 16.5, 16.4; 1000 steps of 80 x 60 (420) at 1, 2: 9.9, 11.9.
int tower_chains(long nchain) {
  if (const char* env = getenv("SF2D_TOWER_CHAINS")) return std::max(1, std::min(4096, atoi(env)));
  return (int)std::max(1L, std::min(16L, (nchain + 4095) / 4096));
}

bool cut_towers(const std::vector<TowerChain>& column, int want, std::vector<Tower>& out) {
  const int n = (int)column.size();
  const int ne = n ? column[0].ne : 0;
  auto follows = [&](const TowerRow& a, const TowerRow& b) {  // b one constant step above a
    return b.inner == a.inner + 4 * ne - 1 && b.left == a.left + 1 && b.right == a.right + 1;
  };
  for (int c = 0; c < n; c++) {
    const TowerRow* r = column[c].row;
    if (column[c].ne != ne || !follows(r[1], r[2]) || !follows(r[2], r[3])) return false;
  }
  for (int c0 = 0; c0 < n;) {
    int c1 = c0 + 1;
    while (c1 < n && column[c1].e0 == column[c1 - 1].e0 + ne && follows(column[c1 - 1].row[3], column[c1 - 1].row[4]) &&
           follows(column[c1 - 1].row[4], column[c1].row[1]))
      c1++;
    const int len = c1 - c0, parts = (len + want - 1) / want;
    for (int p = 0; p < parts; p++) {
      const int a = c0 + (int)((long)len * p / parts), b = c0 + (int)((long)len * (p + 1) / parts);
      out.push_back({column[a].e0, b - a, ne, column[a].row[0], column[a].row[1], column[b - 1].row[NGLL - 1]});
    }
    c0 = c1;
  }
  return true;
}

bool chain_towers(const std::vector<int>& above, const std::vector<TowerChain>& chains, const std::vector<char>& kind,
                  std::vector<Tower>& out, int nshot) {
  const int n = (int)chains.size();
  std::vector<char> has_below(n, 0);
  for (int a : above)
    if (a >= 0) has_below[a] = 1;
  const int want = tower_chains((long)n * nshot);
  std::vector<Tower> towers;
  std::vector<std::pair<int, int>> order;  // height of the tower in its column, tower
  std::vector<TowerChain> column;
  int seen = 0;
  for (int q = 0; q < n; q++) {
    if (has_below[q]) continue;
    int level = 0;
    for (int t = q; t >= 0;) {
      column.clear();
      for (; t >= 0 && kind[t] == CHAIN_STACKED; t = above[t], seen++) column.push_back(chains[t]);
      if (column.empty()) {
        if (kind[t] == CHAIN_ALONE) column.push_back(chains[t]);
        t = above[t];
        seen++;
      }
      if (!cut_towers(column, want, towers)) return false;
      while (order.size() < towers.size()) order.push_back({level++, (int)order.size()});
    }
  }
  if (seen != n) return false;  // a closed ring of chains has no bottom
  std::stable_sort(order.begin(), order.end(), [](auto& a, auto& b) { return a.first < b.first; });
  for (auto& o : order) out.push_back(towers[o.second]);
  return true;
}

void TowerPlan::release() {
  device_free(d_desc); device_free(d_row); device_free(d_id); device_free(d_s01); device_free(d_s23);
  device_free(d_spml); device_free(d_flag);
  *this = TowerPlan();
}

bool build_tower_plan(TowerPlan& P, const std::vector<Tower>& towers, int nglob, const std::vector<uint8_t>& flag,
                      const std::vector<int>& pml_ids, const std::vector<int>& rank, size_t slot_bytes, size_t more_bytes) {
  P.release();
  const int nt = (int)towers.size();
  std::vector<int4> desc((size_t)4 * nt);
  for (int t = 0; t < nt; t++) {
    const Tower& w = towers[t];
    desc[4 * t] = make_int4(w.e0, w.nch, w.ne, P.nrow);
    const TowerRow r[3] = {w.first, w.second, w.top};
    for (int k = 0; k < 3; k++) desc[4 * t + 1 + k] = make_int4(r[k].inner - 1, r[k].left, r[k].right, 0);
    P.nrow += 4 * w.nch + 1;
  }
  auto junction = [&](const Tower& w, int r) { return r % 4 == 0 && r > 0 && r < 4 * w.nch; };
  // how many towers (or chains of them) and layer elements hold each point
  std::vector<uint8_t> cnt((size_t)nglob, 0), npml((size_t)(pml_ids.empty() ? 0 : nglob), 0), two((size_t)nglob, 0);
  for (const Tower& w : towers)
    for (int r = 0; r <= 4 * w.nch; r++) {
      const TowerRow q = w.at(r);
      for (int x = 0; x < 4 * w.ne - 1; x++) cnt[q.inner + x]++;
      cnt[q.left]++;
      cnt[q.right]++;
      if (junction(w, r)) {
        two[q.left]++;
        two[q.right]++;
      }
    }
  for (int g : pml_ids) npml[g]++;
  P.is_if.assign((size_t)nglob, 0);
  std::vector<int> idx((size_t)nglob, -1), order, order4, orderp;
  for (int g = 0; g < nglob; g++) {
    const int np = pml_ids.empty() ? 0 : npml[g];
    if (np == 0 && cnt[g] <= 1 && !flag[g]) continue;
    const int n = cnt[g] + two[g];
    if (n > 4 || np > 4) {
      P.release();
      return false;
    }
    P.is_if[g] = 1;
    (np ? orderp : n > 2 ? order4 : order).push_back(g);
  }
  P.n2 = (int)order.size();
  order.insert(order.end(), order4.begin(), order4.end());
  P.n4 = (int)order.size();
  order.insert(order.end(), orderp.begin(), orderp.end());
  P.n = (int)order.size();
  for (int q = 0; q < P.n; q++) idx[order[q]] = q;
  struct Share { int rank, slot; };
  std::vector<Share> share((size_t)4 * P.n, Share{0, -1});
  std::vector<int4> row((size_t)P.nrow);
  int ns = 0, nr = 0;
  auto give = [&](int g, int rk) {  // a slot for point g, kept in the order of the ranks
    Share* s = &share[(size_t)4 * idx[g]];
    int k = 0;
    while (s[k].slot >= 0) k++;
    for (; k > 0 && s[k - 1].rank > rk; k--) s[k] = s[k - 1];
    s[k] = {rk, ns++};
  };
  for (const Tower& w : towers)
    for (int r = 0; r <= 4 * w.nch; r++) {
      const TowerRow t = w.at(r);
      const int c = std::min(r / 4, w.nch - 1);
      const int rk = rank[w.e0 + c * w.ne];
      unsigned long long m = 0ull;
      const int first = ns;
      auto take = [&](int x, int g) {
        if (!P.is_if[g]) return;
        m |= 1ull << x;
        give(g, rk);
      };
      take(0, t.left);
      for (int x = 1; x < 4 * w.ne; x++) take(x, t.inner + x - 1);
      take(4 * w.ne, t.right);
      const int second = ns;
      if (junction(w, r)) {
        const int below = rank[w.e0 + (c - 1) * w.ne];
        if (P.is_if[t.left]) give(t.left, below);
        if (P.is_if[t.right]) give(t.right, below);
      }
      row[nr++] = make_int4((int)(unsigned)(m & 0xffffffffull), (int)(unsigned)(m >> 32), first, second);
    }
  P.nslot = ns;
  const size_t point_bytes = sizeof(int) + 2 * sizeof(int2) + sizeof(uint8_t);
  if (desc.size() * sizeof(int4) + row.size() * sizeof(int4) + (size_t)P.n * point_bytes +
          (size_t)(P.n - P.n4) * sizeof(int4) + (size_t)ns * slot_bytes + more_bytes > spare_memory()) {
    P.release();
    return false;
  }
  std::vector<int2> s01((size_t)P.n), s23((size_t)(P.n - P.n2));
  for (int q = 0; q < P.n; q++) {
    const Share* s = &share[(size_t)4 * q];
    s01[q] = make_int2(s[0].slot, s[1].slot);
    if (q >= P.n2) s23[q - P.n2] = make_int2(s[2].slot, s[3].slot);
  }
  std::vector<int4> spml((size_t)(P.n - P.n4), make_int4(-1, -1, -1, -1));
  for (size_t k = 0; k < pml_ids.size(); k++) {
    int4& p = spml[idx[pml_ids[k]] - P.n4];
    int* sl[4] = {&p.x, &p.y, &p.z, &p.w};
    int m = 0;
    while (*sl[m] >= 0) m++;
    *sl[m] = (int)k;
  }
  std::vector<uint8_t> fl((size_t)P.n);
  for (int q = 0; q < P.n; q++) fl[q] = flag[order[q]];
  P.ntower = nt;
  P.d_desc = device_copy(desc.data(), desc.size());
  P.d_row = device_copy(row.data(), row.size());
  P.d_id = device_copy(order.data(), order.size());
  P.d_s01 = device_copy(s01.data(), s01.size());
  P.d_s23 = device_copy(s23.data(), s23.size());
  P.d_spml = device_copy(spml.data(), spml.size());
  P.d_flag = device_copy(fl.data(), fl.size());
  return true;
}

void tower_release(Mesh* mp) {
  TowerState* T = mp->tower;
  if (!T) return;
  batch_drop_graph(mp);
  T->plan.release();
  device_free(T->d_slot);
  device_free(T->d_layer);
  device_free(T->d_store);
  for (int s = 0; s < 2; s++) {
    device_free(T->d_other[s]);
    device_free(T->d_acc[s]);
  }
  delete T;
  mp->tower = nullptr;
}

// whether every point inside a tower has one inverse mass for both components (rmassx, rmassz: caller's numbering)
bool tower_masses_fit(const Mesh* mp, const float* rmassx, const float* rmassz) {
  for (int g = 0; g < mp->nglob; g++)
    if (rmassx[g] != rmassz[g]) {
      const int id = mp->point_id.empty() ? g : mp->point_id[g];
      if (id < mp->nglob_el && !mp->tower->plan.is_if[id]) return false;
    }
  return true;
}

}  // namespace sf2d

using namespace sf2d;

extern "C" {

int sf2d_tower_prepare(long* Mesh_pointer, const float* rmassx, const float* rmassz) {
  Mesh* mp = handle(Mesh_pointer);
  tower_release(mp);
  if (!mp->chain || (!mp->first_touch && mp->simulation_type == 1) || !mp->d_col_rows || mp->assembly != 0 ||
      mp->anisotropy || getenv("SF2D_NO_TOWERS"))
    return 0;
  const int npatch = mp->npatch, ng = mp->nglob;
  const std::vector<int4>& rows = mp->h_col_rows;
  const std::vector<int>& ends = mp->h_col_ends;
  const std::vector<int>& pd = mp->h_patch_desc;
  if ((int)mp->h_above.size() != npatch || (int)ends.size() != npatch * NGLL) return 0;
  // a chain all of whose elements belong to the CPML layer has no force of its own
  std::vector<TowerChain> chains(npatch);
  std::vector<char> kind(npatch, CHAIN_STACKED);
  std::vector<int> rank((size_t)mp->nspec, 0);  // descriptors lie colour by colour
  std::vector<char> source((size_t)mp->nspec, 0);
  for (int e : mp->h_src_ispec) source[e] = 1;
  if (mp->simulation_type == 3)
    for (int e : mp->h_rec_ispec) source[e] = 1;  // adjoint sources
  for (int q = 0; q < npatch; q++) {
    TowerChain& c = chains[q];
    c.e0 = pd[4 * q];
    c.ne = pd[4 * q + 3] & 0xf;
    for (int j = 0; j < NGLL; j++) {
      const int4 r = rows[(size_t)q * NGLL + j];
      c.row[j] = {r.x + 1, r.y, ends[(size_t)q * NGLL + j]};
    }
    rank[c.e0] = q;
    // a chain with a source starts and ends at interface rows, so that the source's force comes first in the sum
    bool layer = true, alone = false;
    for (int k = 0; k < c.ne; k++) {
      const int e = mp->ispec_of_pos[c.e0 + k];
      layer = layer && pml_element(mp, e);
      alone = alone || source[e];
    }
    if (layer) kind[q] = CHAIN_SKIP;
    else if (alone) kind[q] = CHAIN_ALONE;
  }
  std::vector<Tower> towers;
  if (!chain_towers(mp->h_above, chains, kind, towers, mp->batch ? mp->batch->nshot : 1)) return 0;
  // points that something besides the towers acts on or looks at
  std::vector<uint8_t> flag((size_t)ng, 0);
  auto mark_element = [&](int ispec, uint8_t f) {
    const int* ib = mp->h_chain_ids.data() + (size_t)mp->pos_of_ispec[ispec] * NGLL2;
    for (int p = 0; p < NGLL2; p++) flag[ib[p]] |= f;
  };
  auto dev = [&](int g) { return mp->point_id.empty() ? g : mp->point_id[g]; };
  auto solid = [&](int e) { return mp->h_is_acoustic.empty() || !mp->h_is_acoustic[e]; };
  for (int e : mp->h_src_ispec)
    if (solid(e)) mark_element(e, IF_ACC);
  for (int e : mp->h_rec_ispec)
    if (solid(e)) mark_element(e, IF_LOOKED_AT);
  for (int g : mp->h_stacey_points) flag[g] |= IF_ACC;
  for (int g : mp->h_uncovered_points)
    if (g < mp->nglob_el) flag[g] |= IF_ACC;
  for (int g : mp->h_coupling_points) flag[dev(g)] |= IF_ACC;
  const std::vector<int>& pml = pml_point_ids(mp, false);
  for (int g : pml) flag[g] |= IF_PML;
  for (int g : mp->h_pml_points) flag[g] |= IF_PML_EDGE;
  for (int g : mp->h_coupling_points)
    if (flag[dev(g)] & IF_PML_EDGE) flag[dev(g)] |= IF_KEEP;
  for (int g = 0; g < ng; g++)
    if (rmassx[g] != rmassz[g]) flag[dev(g)] |= IF_LOOKED_AT;
  for (int g = mp->nglob_el; g < ng; g++) flag[g] = 0;  // no solid element has these
  TowerState* T = new TowerState();
  const int nshot = mp->simulation_type == 3 ? 2 : mp->batch && mp->batch->ps == 1 ? mp->batch->nshot : 1;
  if (!build_tower_plan(T->plan, towers, ng, flag, pml, rank, nshot * sizeof(float2), pml.size() * sizeof(float2))) {
    delete T;
    return 0;
  }
  if (!pml.empty()) T->d_layer = device_alloc<float2>(pml.size());
  T->geo = tower_geometry(mp);
  mp->tower = T;
  if (!reserve_slots(mp, nshot)) tower_release(mp);
  return mp->tower != nullptr;
}

int sf2d_tower_ready(long* Mesh_pointer) { return handle(Mesh_pointer)->tower != nullptr; }

void sf2d_tower_begin(long* Mesh_pointer) {
  Mesh* mp = handle(Mesh_pointer);
  if (!mp->tower) fail("sf2d_tower_begin: no towers");
  clear_interface(mp, (float2*)mp->d_accel, 0, 1);
}

void sf2d_tower_step(long* Mesh_pointer, int it, int last, int checkpoint, float* absorb, float deltat,
                     float deltatsqover2, float deltatover2) {
  Mesh* mp = handle(Mesh_pointer);
  if (!mp->tower || !mp->accel_partial || mp->pending_corrector[0])
    fail("sf2d_tower_step: call after update_displacement_cuda and sf2d_tower_begin");
  if (it < 1 || it > mp->nstep) fail("sf2d_tower_step: it=%d outside 1..%d", it, mp->nstep);
  float2 *d = (float2*)mp->d_displ, *v = (float2*)mp->d_veloc;
  float2* const r = checkpoint >= 0 ? (float2*)grad_checkpoint_inputs(mp, checkpoint) : nullptr;
  const TowerFields F{d, v, d, v, r, (float2*)mp->d_accel, 0, 1, last ? 1 : 0};
  // displacement of the receivers in solid elements; the fluid records its own, and the caller the run's last step
  const int record = !last && mp->nrec_local > 0 && mp->h_seismotype[0] == 1;
  if (record && it > mp->nlength_seismogram) fail("sf2d_tower_step: step %d after the seismograms' last", it);
  TowerState* T = mp->tower;
  float2* store = nullptr;
  if (absorb && mp->stacey && mp->num_abs > 0) {
    prepare_store(mp, mp->nstep);
    if (T->store_first < 0) T->store_first = it;
    store = T->d_store + store_points(mp) * (it - T->store_first);
  }
  launch_tower(mp, F, it, record ? mp->d_seismo[0] : nullptr, 0, nullptr, {deltatover2, deltat, deltatsqover2}, true,
               nullptr, store);
  if (store && (last || it - T->store_first + 1 == T->store_steps)) {
    const int n = it - T->store_first + 1;
    check_hip(hipMemcpyAsync(absorb - 2 * store_points(mp) * (n - 1), T->d_store, store_points(mp) * n * sizeof(float2),
                             hipMemcpyDeviceToHost, mp->stream),
              "Stacey terms D2H");
    check_hip(hipStreamSynchronize(mp->stream), "sf2d_tower_step");
    T->store_first = -1;
  }
  if (last) mp->accel_partial = 0;
}

int sf2d_tower_adjoint_begin(long* Mesh_pointer) {
  Mesh* mp = handle(Mesh_pointer);
  TowerState* T = mp->tower;
  if (!T || mp->simulation_type != 3) fail("sf2d_tower_adjoint_begin: no towers, or not SIMULATION_TYPE = 3");
  if (!T->d_acc[1] && 4 * (size_t)mp->nglob * sizeof(float2) > spare_memory()) return 0;
  for (int s = 0; s < 2; s++) {
    if (!T->d_other[s]) T->d_other[s] = device_alloc<float>((size_t)2 * mp->nglob);
    if (!T->d_acc[s]) T->d_acc[s] = device_zeros<float2>((size_t)mp->nglob);
  }
  if (mp->stacey) prepare_store(mp, mp->nstep);
  T->store_first = -1;
  return 1;
}

void sf2d_tower_adjoint_step(long* Mesh_pointer, int it, int last, const float* absorb, float deltat,
                             float deltatsqover2, float deltatover2, float b_deltat, float b_deltatsqover2,
                             float b_deltatover2) {
  Mesh* mp = handle(Mesh_pointer);
  TowerState* T = mp->tower;
  if (!T || !T->d_other[0] || mp->pending_corrector[0] || mp->pending_corrector[1])
    fail("sf2d_tower_adjoint_step: call after update_displacement_cuda and sf2d_tower_adjoint_begin");
  if (it < 1 || it > mp->nstep) fail("sf2d_tower_adjoint_step: it=%d outside 1..%d", it, mp->nstep);
  const TowerPlan& P = T->plan;
  const int sample = mp->nstep - it;  // 0-based time sample of the forward run
  const size_t np = store_points(mp);
  const bool edges = mp->stacey && mp->num_abs > 0;
  if (edges && (T->store_first < 0 || sample < T->store_first)) {
    T->store_first = std::max(0, sample + 1 - T->store_steps);
    check_hip(hipMemcpyAsync(T->d_store, absorb + 2 * np * T->store_first,
                             np * (sample + 1 - T->store_first) * sizeof(float2), hipMemcpyHostToDevice, mp->stream),
              "Stacey terms H2D");
  }
  float2 *d0 = (float2*)mp->d_displ, *v0 = (float2*)mp->d_veloc, *d1 = (float2*)mp->d_b_displ, *v1 = (float2*)mp->d_b_veloc;
  const PairFields F{d0, v0, d1, v1, (float2*)T->d_other[0], v0, (float2*)mp->d_accel, (float2*)T->d_other[1], v1,
                     (float2*)mp->d_b_accel,
                     T->d_acc[0], T->d_acc[1], {deltatover2, deltat, deltatsqover2},
                     {b_deltatover2, b_deltat, b_deltatsqover2}, 2, last ? 1 : 0};
  PairEdges E{};
  E.faces = stacey_faces(mp);
  E.receivers = receiver_set(mp);
  E.sources = source_set(mp);
  E.it = sample;
  E.cur = it - 1;
  E.nstep = mp->nstep;
  E.nface_wg = edges ? (mp->num_abs * NGLL + 63) / 64 : 0;
  E.nsource = mp->nsources_local;
  E.nadj = mp->nadj_rec_local;
  E.nreceiver = last ? 0 : mp->nrec_local;
  E.adj = mp->d_source_adjoint;
  E.store = edges ? T->d_store + np * (sample - T->store_first) : nullptr;
  E.seismo = mp->d_seismo[0];
  if (E.nreceiver > 0 && it > mp->nlength_seismogram) fail("sf2d_tower_adjoint_step: step %d after the last sample", it);
  float2* const slot = tower_slots(T, 2);
  using K = decltype(&k_tower<0, 0, PairFields, PairEdges>);
  const K kern[5] = {k_tower<0, 0, PairFields, PairEdges>, k_tower<1, 0, PairFields, PairEdges>,
                     k_tower<2, 0, PairFields, PairEdges>, k_tower<3, 0, PairFields, PairEdges>,
                     k_tower<4, 0, PairFields, PairEdges>};
  launch_k_tower(mp, kern[mp->tower->geo], F, E, slot, F.nm0);
  if (P.n > 0) {
    hipLaunchKernelGGL(k_interface_pair, dim3((P.n + IF_T - 1) / IF_T, 2), dim3(IF_T), 0, mp->stream, interface_args(P), slot,
                       P.nslot, F, mp->d_rmassx, mp->d_rmassz);
    check_hip(hipGetLastError(), "k_interface_pair launch");
  }
  launch_kernels(mp, mp->d_displ, mp->d_accel, mp->d_b_displ);
  if (last) return;
  std::swap(mp->d_displ, T->d_other[0]);
  std::swap(mp->d_b_displ, T->d_other[1]);
}

}  // extern "C"
