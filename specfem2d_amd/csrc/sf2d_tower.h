// Towers of chains and the interface between them: the plan that the fused time steps of the solid (tower.hip) and of
// the fluid (acoustic.hip) share.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "sf2d_device.h"
#include "sf2d_mesh.h"

namespace sf2d {

// flags of an interface point
constexpr uint8_t IF_ACC = 1;        // boundary terms arrive in the step's accumulator
constexpr uint8_t IF_PML = 2;        // CPML layer point: keeps its previous-step field
constexpr uint8_t IF_PML_EDGE = 4;   // on the layer's outer boundary
constexpr uint8_t IF_KEEP = 8;       // solid: an edge point on a fluid-solid edge, cleared after the fluid has read it
constexpr uint8_t IF_FREE = 16;      // fluid: free surface
constexpr uint8_t IF_COUPLED = 32;   // fluid: on a fluid-solid edge, the solid reads its acceleration
constexpr uint8_t IF_LOOKED_AT = 64; // something reads the point during the step

// GLL row of a tower: id of x = 1 (the inner points are consecutive), of x = 0 and of x = 4 ne
struct TowerRow {
  int inner, left, right;
};

struct Tower {
  int e0, nch, ne;  // first element position (consecutive upwards), chains, elements per chain
  TowerRow first, second, top;  // rows 0 and 1 and the topmost; rows from 1 to the last but one go up in constant steps
  TowerRow at(int r) const {
    if (r == 0) return first;
    if (r == 4 * nch) return top;
    return {second.inner + (r - 1) * (4 * ne - 1), second.left + r - 1, second.right + r - 1};
  }
};

// cuts a column of chains into towers of at most `want` chains (about equal ones) whose rows fit Tower; false when the
// inner rows of some chain do not go up in constant steps
struct TowerChain {
  int e0, ne;
  TowerRow row[NGLL];
};
bool cut_towers(const std::vector<TowerChain>& column, int want, std::vector<Tower>& out);
int tower_chains(long nchain);
// the towers of chains (above: the chain on top of each, -1: none), the lowest of all columns first, so that neighbours
// run together.  kind: CHAIN_ALONE a tower of its own, CHAIN_SKIP none (the chain has no force of its own)
enum : char { CHAIN_STACKED, CHAIN_ALONE, CHAIN_SKIP };
bool chain_towers(const std::vector<int>& above, const std::vector<TowerChain>& chains, const std::vector<char>& kind,
                  std::vector<Tower>& out, int nshot = 1);

struct TowerPlan {
  int ntower = 0, nrow = 0;
  // [ntower][4] {first element position, chains, elements per chain, first row record}, {id of x = 1 less one, id of
  // x = 0, id of x = 4 ne, -} of row 0, of row 1 and of the topmost row
  int4* d_desc = nullptr;
  int4* d_row = nullptr;      // [nrow] {mask low, mask high, first slot, first split slot} per GLL row, bottom to top;
                              // mask bit x: point x of the row is an interface point
  int nslot = 0;              // slots of the towers; the CPML layer's are numbered by element point
  // interface points: [0, n2) have at most two tower slots and none of the layer, [n2, n4) up to four, [n4, n) are points
  // of the CPML layer with up to four tower and four layer slots
  int n = 0, n2 = 0, n4 = 0;
  int* d_id = nullptr;        // [n]
  int2* d_s01 = nullptr;      // [n] tower slots (-1: none)
  int2* d_s23 = nullptr;      // [n - n2]
  int4* d_spml = nullptr;     // [n - n4]
  uint8_t* d_flag = nullptr;  // [n]
  std::vector<char> is_if;    // [nglob]
  void release();
};

// builds the plan over the points of the towers and the flagged ones; pml_ids: point of each CPML element point.  False
// when more than four towers (chains) or layer elements meet in a point.
// The slots of a point are in the order of rank (of the chain at each first element position), and where two chains of a
// tower meet, the interface points of its left and right column take the two chains' forces in slots of their own (the
// lower one's are the row's split slots): the interface then sums a point's forces one chain at a time in the order in
// which a launch per colour adds them.
// False too when the spare memory does not hold the plan, slot_bytes for each slot and more_bytes.
bool build_tower_plan(TowerPlan& P, const std::vector<Tower>& towers, int nglob, const std::vector<uint8_t>& flag,
                      const std::vector<int>& pml_ids, const std::vector<int>& rank, size_t slot_bytes, size_t more_bytes);

constexpr int IF_T = 64;  // threads per workgroup of the interface kernels: one wave, so that few points spread over many CUs

// arguments of the interface kernels
struct InterfaceArgs {
  int n, n2, n4;
  const int* id;
  const int2 *s01, *s23;
  const int4* spml;
  const uint8_t* flag;
};
inline InterfaceArgs interface_args(const TowerPlan& P) {
  return {P.n, P.n2, P.n4, P.d_id, P.d_s01, P.d_s23, P.d_spml, P.d_flag};
}

__device__ __forceinline__ void add_slot(float& r, float p) { r += p; }
__device__ __forceinline__ void add_slot(float2& r, float2 p) {
  r.x += p.x;
  r.y += p.y;
}
// The slots of interface point q (-1: none).  Loaded before anything that depends on them, and their values without
// branches (a missing slot reads slot 0): an interface kernel is a chain of dependent loads, and a branch around each
// would make the chain longer (80 x 60 elements: 4.4 us, 3.2 without).
struct SlotIds {
  int t[4], p[4];
};
__device__ __forceinline__ SlotIds slot_ids(const InterfaceArgs& A, int q) {
  SlotIds s;
  const int2 a = A.s01[q];
  int2 b = make_int2(-1, -1);
  int4 p = make_int4(-1, -1, -1, -1);
  if (q >= A.n2) b = A.s23[q - A.n2];
  if (q >= A.n4) p = A.spml[q - A.n4];
  s.t[0] = a.x; s.t[1] = a.y; s.t[2] = b.x; s.t[3] = b.y;
  s.p[0] = p.x; s.p[1] = p.y; s.p[2] = p.z; s.p[3] = p.w;
  return s;
}
template <typename T>
struct SlotValues {
  T v[4];
};
template <typename T>
__device__ __forceinline__ SlotValues<T> slot_values(bool more, const int (&s)[4], const T* __restrict__ slot) {
  SlotValues<T> r;
#pragma unroll
  for (int k = 0; k < 2; k++) r.v[k] = slot[max(s[k], 0)];
  r.v[2] = r.v[3] = T{};
  if (more) {
#pragma unroll
    for (int k = 2; k < 4; k++) r.v[k] = slot[max(s[k], 0)];
  }
  return r;
}
// r plus the values, in order
template <typename T>
__device__ __forceinline__ T sum_slots(const int (&s)[4], const SlotValues<T>& x, T r) {
#pragma unroll
  for (int k = 0; k < 4; k++) {
    T n = r;
    add_slot(n, x.v[k]);
    if (s[k] >= 0) r = n;
  }
  return r;
}

struct Newmark {
  float dto2, dt, dt2o2;
};

// fluid-solid edge points: ids, normals out of the fluid, weights (compute_coupling_acoustic_el.f90:34-150,
// compute_coupling_viscoelastic_ac.f90:34-130)
struct CouplingPoints {
  int n;
  const int* id;
  const float2* normal;
  const float* w;
};
// fluid side: pdd += w (u . n); sign -1: the adjoint run's term, u minus the adjoint acceleration (:104-109)
__device__ __forceinline__ void couple_fluid(const CouplingPoints& C, int k, const float2* __restrict__ displ, float sign,
                                             float* __restrict__ pdd) {
  if (k >= C.n) return;
  const int g = C.id[k];
  const float2 u = displ[g], nv = C.normal[k];
  const float dn = (sign * u.x) * nv.x + (sign * u.y) * nv.y;
  atomic_add_f32(&pdd[g], C.w[k] * dn);
}
// solid side: accel += w n p with the fluid pressure p = -pdd; sign -1 and the adjoint potential in place of pdd: the
// adjoint run's pressure p = potential (:98-102)
__device__ __forceinline__ void couple_solid(const CouplingPoints& C, int k, const float* __restrict__ pdd, float sign,
                                             float* __restrict__ accel) {
  if (k >= C.n) return;
  const int g = C.id[k];
  const float pr = sign * -pdd[g];
  const float2 nv = C.normal[k];
  const float wk = C.w[k];
  atomic_add_f32(&accel[2 * (size_t)g], wk * nv.x * pr);
  atomic_add_f32(&accel[2 * (size_t)g + 1], wk * nv.y * pr);
}

// the coupling points and the fluid's acceleration (acoustic.hip); n = 0 without fluid-solid edges
CouplingPoints acoustic_coupling(Mesh* mp, const float** pdd);
// CPML layer in the fused steps (pml.hip): the point of each element point of the solid's or the fluid's layer (packed
// order), the previous-step field [nglob], and the layer's forces into one slot per element point
const std::vector<int>& pml_point_ids(const Mesh* mp, bool fluid);
const std::vector<int>& pml_edge_points(const Mesh* mp, bool fluid);
void* pml_old_field(const Mesh* mp, bool fluid);
void pml_elastic_slots(Mesh* mp, float2* slots);
void pml_acoustic_slots(Mesh* mp, const float* pot, const float* pd, float2* slots);  // {flux term, memory term}

}  // namespace sf2d
