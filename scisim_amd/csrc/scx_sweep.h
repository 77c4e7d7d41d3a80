// scx_sweep.h -- device code shared by the sweep kernels: contact records, relative
// velocities, the local Coulomb solve, the Fischer-Burmeister residual and the kernels'
// arguments. Every sweep kernel updates and evaluates a contact through these functions, and
// FMA contraction is per source expression, so a contact rounds the same way in all of them.
#pragma once

#pragma clang fp contract(on)

#include "scx_device.h"
#include "scx_internal.h"

#include <type_traits>

namespace scx {

template <typename Real>
struct Vec4 {
  using type = double4;
};
template <>
struct Vec4<float> {
  using type = float4;
};

template <int D, typename Real>
struct Rec {
  uint32_t a, b;
  Real n[3], s[3], t[3];
  Real la, lb, wn, wt, mu, f;
};

// The rest of the contact frame from n (and s in 3D): t = n x s (3D), t = (-n_y, n_x) (2D).
template <int D, typename Real>
__device__ __forceinline__ void frame_from_ns(Rec<D, Real>& R) {
  if (D == 3) {
    R.t[0] = R.n[1] * R.s[2] - R.n[2] * R.s[1];
    R.t[1] = R.n[2] * R.s[0] - R.n[0] * R.s[2];
    R.t[2] = R.n[0] * R.s[1] - R.n[1] * R.s[0];
  } else {
    R.t[0] = -R.n[1];
    R.t[1] = R.n[0];
    R.t[2] = 0;
    R.s[0] = R.s[1] = R.s[2] = 0;
    R.la = R.lb = 0;
  }
}

template <int D, typename Real>
__device__ __forceinline__ void load_rec(const ContactSoA<Real>& c, uint32_t k, Rec<D, Real>& R) {
  R.a = c.a[k];
  R.b = c.b[k];
#pragma unroll
  for (int d = 0; d < 3; ++d) R.n[d] = c.n[3 * (size_t)k + d];
  if (D == 3) {
#pragma unroll
    for (int d = 0; d < 3; ++d) R.s[d] = c.s[3 * (size_t)k + d];
    R.la = c.la[k];
    R.lb = c.lb[k];
  }
  frame_from_ns<D, Real>(R);
  R.wn = c.wn[k];
  R.wt = c.wt[k];
  R.mu = c.mu[k];
  R.f = c.forcing[k];
}

// Pre-impulse relative velocity in the contact frame, u = H_a v_a - H_b v_b + w,
// computed in precision T from bodies stored in precision Real.
template <int D, typename T, typename Real>
__device__ __forceinline__ void rel_vel(const Rec<D, Real>& R, const typename Vec4<Real>::type& va,
                                        const typename Vec4<Real>::type& wa, const typename Vec4<Real>::type& vb,
                                        const typename Vec4<Real>::type& wb, T u[3]) {
  const T dv[3] = {(T)va.x - (T)vb.x, (T)va.y - (T)vb.y, (T)va.z - (T)vb.z};
  const T n[3] = {(T)R.n[0], (T)R.n[1], (T)R.n[2]};
  const T t[3] = {(T)R.t[0], (T)R.t[1], (T)R.t[2]};
  u[0] = n[0] * dv[0] + n[1] * dv[1] + n[2] * dv[2] + (T)R.f;
  if (D == 3) {
    const T s[3] = {(T)R.s[0], (T)R.s[1], (T)R.s[2]};
    const T la = (T)R.la, lb = (T)R.lb;
    const T ca[3] = {(T)wa.y * n[2] - (T)wa.z * n[1], (T)wa.z * n[0] - (T)wa.x * n[2],
                     (T)wa.x * n[1] - (T)wa.y * n[0]};
    const T cb[3] = {(T)wb.y * n[2] - (T)wb.z * n[1], (T)wb.z * n[0] - (T)wb.x * n[2],
                     (T)wb.x * n[1] - (T)wb.y * n[0]};
    T uv[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) uv[d] = dv[d] - la * ca[d] - lb * cb[d];
    u[1] = s[0] * uv[0] + s[1] * uv[1] + s[2] * uv[2];
    u[2] = t[0] * uv[0] + t[1] * uv[1] + t[2] * uv[2];
  } else {
    u[1] = t[0] * dv[0] + t[1] * dv[1];
    u[2] = 0;
  }
}

// Exact Coulomb solution for the block diag(w_n, w_t, w_t): separate, stick, or slide
// on the cone boundary against the tangential pre-velocity.
template <int D, typename Real>
__device__ __forceinline__ void local_solve(const Rec<D, Real>& R, const Real u[3], const Real r[3], Real rn[3]) {
  const Real bn = u[0] - R.wn * r[0];
  const Real n0 = -bn / R.wn;
  if (!(n0 > (Real)0)) {
    rn[0] = rn[1] = rn[2] = 0;
    return;
  }
  rn[0] = n0;
  Real nrm2 = 0;
#pragma unroll
  for (int a = 1; a < D; ++a) {
    rn[a] = -(u[a] - R.wt * r[a]) / R.wt;
    nrm2 += rn[a] * rn[a];
  }
  if (D == 2) rn[2] = 0;
  const Real lim = R.mu * n0;
  // (2D: the root of a rounded square is the number's size, up to the range's ends)
  const Real nrm = D == 2 ? fabs(rn[1]) : sqrt(nrm2);
  if (nrm > lim) {
    const Real sc = (nrm > (Real)0) ? lim / nrm : (Real)0;
#pragma unroll
    for (int a = 1; a < D; ++a) rn[a] *= sc;
  }
}

// FB residual of one contact (De Saxce change of variable), ||phi||^2, in precision T
// (FP64 for every decision on the tolerance; FP32 only for the estimate of the FP32 phase).
template <int D, typename T = double>
__device__ __forceinline__ T fb_err(T mu, const T* r, const T* u) {
  T uT2 = (T)0;
#pragma unroll
  for (int a = 1; a < D; ++a) uT2 += u[a] * u[a];
  const T un_hat = u[0] + mu * (D == 2 ? fabs(u[1]) : sqrt(uT2));  // (2D as in local_solve)
  T xh[3], yh[3];
  xh[0] = mu * r[0];
  yh[0] = un_hat;
#pragma unroll
  for (int a = 1; a < D; ++a) {
    xh[a] = r[a];
    yh[a] = mu * u[a];
  }
  T z0 = (T)0;
#pragma unroll
  for (int a = 0; a < D; ++a) z0 += xh[a] * xh[a] + yh[a] * yh[a];
  T z1[2] = {(T)0, (T)0}, nz1 = (T)0;
#pragma unroll
  for (int a = 1; a < D; ++a) {
    z1[a - 1] = (T)2 * (xh[0] * xh[a] + yh[0] * yh[a]);
    nz1 += z1[a - 1] * z1[a - 1];
  }
  nz1 = D == 2 ? fabs(z1[0]) : sqrt(nz1);
  const T s1 = sqrt(z0 + nz1);
  const T s2 = sqrt(fmax((T)0, z0 - nz1));
  T e = xh[0] + yh[0] - (T)0.5 * (s1 + s2);
  e = e * e;
#pragma unroll
  for (int a = 1; a < D; ++a) {
    const T dir = !(nz1 > (T)0) ? (T)0 : D == 2 ? copysign((T)1, z1[0]) : z1[a - 1] / nz1;
    const T p = xh[a] + yh[a] - (T)0.5 * (s1 - s2) * dir;
    e += p * p;
  }
  // a NaN residual (e.g. from non-finite velocities) counts as infinitely far from the
  // solution: the max reductions drop NaN operands, so it must never read as converged
  return __builtin_isnan(e) ? (T)INFINITY : e;
}

// Body records per slot: 2D one vector [v (3) | minv], 3D two adjacent vectors
// [v (3) | minv][omega (3) | Iinv].
template <int D>
constexpr int kBodyVecs = (D == 3) ? 2 : 1;

template <typename Real>
struct GSArgs {
  ContactSoA<Real> c;
  Real* body;               // body records by slot
  const uint32_t* sid;      // slot -> body id (nullptr: identity)
  const double* v0;         // dim per body
  const double* w0;         // 3 per body (3D)
  uint32_t nbodies;
  uint32_t C;
  const uint32_t* coloff;   // colour offsets
  Real* rbest;              // 3 per contact
  double* partial;          // per-workgroup residual partials
  StepCounters* ctr;
  uint32_t* bar;             // grid barrier state
  uint32_t max_iters;
  uint32_t eval_every;
  double tol;
  int phase;                // 0: only phase, 1: FP32 phase, 2: FP64 polish after FP32
  int apply_init;           // reset velocities to v0 and apply the records' impulses
  uint32_t* lmap;           // per body slot: owning endpoint in the LDS solve (all ones when idle)
  uint32_t tail_col;        // colours [tail_col, ncolours) are swept by workgroup 0 alone (small)
  // ensembles (else cscene == nullptr): per contact (colour order) its scene; per scene the
  // residual of the last evaluations (max ||FB||^2 bits; k_gs uses two buffers in turn,
  // k_gs_flow three) and the sweep at which it met the tolerance (kNoBody until then). A scene
  // that meets the tolerance is frozen: its contacts are skipped until the solve ends.
  const uint32_t* cscene;
  unsigned long long* scene_acc;  // 3 x nscenes
  uint32_t* scene_sweeps;         // nscenes
  uint32_t nscenes;
  // ensembles: the contacts of scenes not yet frozen, compacted colour by colour once
  // enough scenes have frozen (two lists of C entries, alternately rebuilt), and per-colour
  // per-workgroup counts for the compaction (kMaxColours x gridDim); nullptr: no compaction
  uint32_t* act_idx;
  uint32_t* act_part;
  // FP32 phase of one scene: contacts whose residual at the last full evaluation was at
  // least the capture threshold (up to kViolCap, in any order; counts of the two last
  // evaluations, double-buffered), and the word through which workgroup 0 tells the others
  // that one of them is still above the stopping value (nullptr: every sweep is evaluated)
  uint32_t* viol;  // 2 counts, then kViolCap contacts
  uint32_t* vflag;
  // One scene with coherent passes on several workgroups: colours [comp_col, ncolours) are
  // swept as connected components (contacts linked through shared bodies), every component
  // by one workgroup through its L2. comp_parent: per body slot, its parent in a union-find
  // forest over the bodies of those contacts; comp_cnt: an overflow flag, then per
  // workgroup the number of contacts it was given; comp_list: per workgroup kCompCap
  // contacts. comp_parent == nullptr: no component phase.
  uint32_t* comp_parent;
  uint32_t* comp_cnt;
  uint32_t* comp_list;
  uint32_t comp_col;
  int comp_lds;  // hold a workgroup's components in LDS when they fit (else through its L2)
};

// A contact's record and impulse, loaded ahead of its colour pass. Only the thread that
// updates a contact ever writes its impulse, and the record is read-only during the
// solve, so the load may be issued before the grid barrier that opens the pass.
template <int D, typename Real>
struct Loaded {
  Rec<D, Real> R;
  Real r[3];
};

// One contact of a colour pass from its loaded record, on body vectors ia and ib (3D: ia + 1
// and ib + 1 are the angular halves of the same records) read and written through ld/st,
// the new impulse stored through st_r(d, x). rbest: first store the contact's impulse as it
// was before this sweep there (the previous sweep's iterate was the best one so far). Every
// update of a contact goes through this code, wherever its bodies are held.
template <int D, typename Real, typename Ld, typename St, typename StR>
__device__ __forceinline__ void update_core(const Loaded<D, Real>& L, bool init, Real* rbest, size_t ia, size_t ib,
                                            Ld&& ld, St&& st, StR&& st_r) {
  using V = typename Vec4<Real>::type;
  const Rec<D, Real>& R = L.R;
  const bool hasb = R.b != kNoBody;
  V va = ld(ia), wa = {0, 0, 0, 0}, vb = {0, 0, 0, 0}, wb = {0, 0, 0, 0};
  if (D == 3) wa = ld(ia + 1);
  if (hasb) {
    vb = ld(ib);
    if (D == 3) wb = ld(ib + 1);
  }
  const Real r[3] = {L.r[0], L.r[1], L.r[2]};
  if (rbest) {
    rbest[0] = r[0];
    rbest[1] = r[1];
    rbest[2] = r[2];
  }
  Real dr[3];
  if (init) {
    dr[0] = r[0];
    dr[1] = r[1];
    dr[2] = r[2];
  } else {
    Real u[3], rn[3];
    rel_vel<D, Real, Real>(R, va, wa, vb, wb, u);
    local_solve<D, Real>(R, u, r, rn);
    dr[0] = rn[0] - r[0];
    dr[1] = rn[1] - r[1];
    dr[2] = rn[2] - r[2];
    st_r(0, rn[0]);
    st_r(1, rn[1]);
    if (D == 3) st_r(2, rn[2]);
  }
  Real Pi[3];  // the impulse increment in world coordinates
#pragma unroll
  for (int d = 0; d < 3; ++d) Pi[d] = R.n[d] * dr[0] + R.t[d] * dr[D - 1] + ((D == 3) ? R.s[d] * dr[1] : (Real)0);
  va.x += va.w * Pi[0];
  va.y += va.w * Pi[1];
  va.z += va.w * Pi[2];
  st(ia, va);
  Real tau[3];
  if (D == 3) {
#pragma unroll
    for (int d = 0; d < 3; ++d) tau[d] = dr[1] * R.t[d] - dr[2] * R.s[d];
    const Real ka = -R.la * wa.w;
    wa.x += ka * tau[0];
    wa.y += ka * tau[1];
    wa.z += ka * tau[2];
    st(ia + 1, wa);
  }
  if (hasb) {
    vb.x -= vb.w * Pi[0];
    vb.y -= vb.w * Pi[1];
    vb.z -= vb.w * Pi[2];
    st(ib, vb);
    if (D == 3) {
      const Real kb = R.lb * wb.w;
      wb.x -= kb * tau[0];
      wb.y -= kb * tau[1];
      wb.z -= kb * tau[2];
      st(ib + 1, wb);
    }
  }
}

template <typename Real>
struct Vec2 {
  using type = double2;
};
template <>
struct Vec2<float> {
  using type = float2;
};

// Packed record fields, four Reals to a group, group-major over the contacts so that a wave
// reads whole lines: 3D [n | la] [s | lb] [wn wt mu f] [1/m_a 1/m_b 1/I_a 1/I_b],
// 2D [n.x n.y wn wt] [mu f 1/m_a 1/m_b]. The inverse masses ride with the contact, so that a
// body that passes from contact to contact is its velocities alone (2D 2, 3D 6 Reals).
template <int D>
constexpr int kRecGroups = (D == 3) ? 4 : 2;

// The record as load_rec builds it (a and b: only whether b is a body matters), and the
// inverse masses and inertias of a and b.
template <int D, typename Real>
__device__ __forceinline__ void unpack_rec(const typename Vec4<Real>::type* g, bool hasb, Rec<D, Real>& R, Real* im) {
  R.a = 0;
  R.b = hasb ? 0u : kNoBody;
  if constexpr (D == 3) {
    R.n[0] = g[0].x, R.n[1] = g[0].y, R.n[2] = g[0].z, R.la = g[0].w;
    R.s[0] = g[1].x, R.s[1] = g[1].y, R.s[2] = g[1].z, R.lb = g[1].w;
    R.wn = g[2].x, R.wt = g[2].y, R.mu = g[2].z, R.f = g[2].w;
    im[0] = g[3].x, im[1] = g[3].y, im[2] = g[3].z, im[3] = g[3].w;
  } else {
    R.n[0] = g[0].x, R.n[1] = g[0].y, R.n[2] = 0, R.wn = g[0].z, R.wt = g[0].w;
    R.mu = g[1].x, R.f = g[1].y;
    im[0] = g[1].z, im[1] = g[1].w, im[2] = im[3] = 0;
  }
  frame_from_ns<D, Real>(R);
}

template <int D, typename Real>
__device__ __forceinline__ void pack_rec(const Rec<D, Real>& R, const typename Vec4<Real>::type* body, uint32_t C,
                                         uint32_t k, typename Vec4<Real>::type* rec) {
  using V = typename Vec4<Real>::type;
  const bool hasb = R.b != kNoBody;
  const V* pa = body + (size_t)kBodyVecs<D> * R.a;
  const V* pb = body + (size_t)kBodyVecs<D> * (hasb ? R.b : R.a);
  const Real ma = pa[0].w, mb = hasb ? pb[0].w : (Real)0;
  if constexpr (D == 3) {
    rec[k] = V{R.n[0], R.n[1], R.n[2], R.la};
    rec[(size_t)C + k] = V{R.s[0], R.s[1], R.s[2], R.lb};
    rec[2 * (size_t)C + k] = V{R.wn, R.wt, R.mu, R.f};
    rec[3 * (size_t)C + k] = V{ma, mb, pa[1].w, hasb ? pb[1].w : (Real)0};
  } else {
    rec[k] = V{R.n[0], R.n[1], R.wn, R.wt};
    rec[(size_t)C + k] = V{R.mu, R.f, ma, mb};
  }
}

// Working memory of the sweeps without barriers (k_gs_flow). Contacts have places: workgroup
// after workgroup, within one in colour order.
constexpr uint32_t kFlowMaxScenes = 2048;  // an ensemble's residuals, in every workgroup's LDS
constexpr uint32_t kFlowTagMax = 1u << 30;  // the tags of a context start over on cleared slots
constexpr int kFlowMaxBlocks = 256;  // one wave reads every workgroup's flag
// Looks after which a wait has run out, once every workgroup is resident: about eight seconds for
// a body in a slot or another workgroup's part, one for a body in LDS. A wait takes microseconds,
// or as long as other processes have the XCD of the waves that are waited for.
constexpr uint32_t kFlowPolls = 1u << 24;
// Slots of side b follow those of side a, the near ones (read on one XCD alone) of both follow
// the far ones, so that no line holds both kinds; kFlowLine consecutive ones fill at least two lines.
constexpr uint32_t kFlowLine = 16;
// Places of C contacts: a line's worth free behind each XCD's.
__host__ __device__ inline uint32_t flow_places(uint32_t C) {
  return (C + kFlowLine - 1) / kFlowLine * kFlowLine + kXcds * kFlowLine;
}
// Where a contact finds a body (FlowBufs::from, fin)
constexpr uint32_t kFlowWrap = 1, kFlowNear = 2, kFlowHome = 4, kFlowColourBits = 6;
static_assert(kMaxColours <= 1 << kFlowColourBits, "a colour's bits");
template <typename Real>
struct FlowBufs {
  Real* rec;          // packed records, by place
  Real* r;            // impulses: 4 (3D) or 2 (2D) Reals per place
  const uint32_t* from;  // per place, 2: where its bodies come from (as k_gs_flow's FlowContact)
  const uint32_t* fin;   // per place, 2: where its bodies are after their last contacts
  const uint32_t* beg;   // per workgroup, kMaxColours + 1: the first place of each colour
  const uint32_t* place;  // of each contact
  const uint32_t* who;   // the contact at each place
  uint32_t* scene;    // per place (ensembles)
  void* slots;        // outbox slots, in 16-byte pieces
  uint32_t xcds;      // XCDs that take part
  uint32_t* flags;    // per workgroup: 2 * tag + whether it holds a contact above the threshold
  void* parts;        // per workgroup: its largest residual and the tag
  uint32_t tag0;      // first tag of this launch: above every tag in slots, flags and parts
  // The FP32 phase's first sweeps skip evaluations by the stopping value, as k_gs does on
  // several workgroups with a tail or a component phase. Elsewhere k_gs evaluates every sweep,
  // so that its stagnation test knows the best residual of those sweeps too, and the
  // threshold here is the best residual from the start.
  int skip_early;
  uint32_t polls;     // looks of a wait for bodies during the sweeps, at most (kFlowPolls but in tests)
  uint32_t home;      // bodies of a workgroup that its LDS holds, and 64 more
  uint32_t rows;      // rows of a workgroup's contacts, at most
  uint32_t kept;      // contacts of a workgroup that its LDS holds
};
struct FlowLinks {
  unsigned long long* mask;  // per body: its colours; entry n: the table's length
  uint32_t* start;           // per body: start of its entries in the table
  uint32_t* where;           // per body: see k_flow_homes
  uint32_t* table;           // each body's contacts in colour order
  uint32_t* own;             // per contact: its workgroup
  uint32_t* place;
  uint32_t* who;
  uint32_t* scene;
  uint32_t* lo;              // per workgroup, kMaxColours + 1: see k_flow_ranges
  uint32_t* beg;
  uint32_t* homes;           // per workgroup: bodies that may live in its LDS
  uint2* from;
  uint2* fin;
};
// first: contacts before those of each first body in the order of the bodies, or null; home: as
// FlowBufs::home.
hipError_t launch_flow_links(scx_ctx* c, uint32_t C, const uint32_t* ca, const uint32_t* cb, const uint32_t* first,
                             const FlowLinks& L, uint32_t xcds, uint32_t per_xcd, uint32_t home);
// Packs the records and launches the sweeps on per_xcd workgroups of each of F.xcds XCDs; *launched is false when a
// cooperative launch is not to be had (nothing ran).
template <int D, typename Real>
hipError_t launch_gs_flow(scx_ctx* c, GSArgs<Real> A, FlowBufs<Real> F, uint32_t per_xcd, bool* launched);

}  // namespace scx
