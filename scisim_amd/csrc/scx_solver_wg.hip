// scx_solver_wg.hip -- the sweeps of a contact set whose touched bodies one workgroup can hold
// in LDS: the velocities live in LDS for the whole solve and the contact records stream from
// the L2 in colour order, loaded one pass ahead, so a colour pass costs LDS traffic and a
// workgroup barrier instead of a grid barrier and coherent gathers.
//
// What bounds it: the latency of one update per colour (about 1.1 us in FP64 3D, most of it the
// dependent chain of divisions and the square root), then the CU's FP64 rate. Measured on
// MI355X against the sweeps it replaces (k_gs), per sweep: 3,347 sphere contacts in 12 colours,
// FP64, residual every 20 sweeps: 87 -> 18.7 us; 2,600 sphere contacts, FP64, residual after
// most sweeps: 72 -> 24 us.
#pragma clang fp contract(on)

#include "scx_device.h"
#include "scx_internal.h"
#include "scx_sweep.h"

#include <algorithm>

namespace scx {

// A contact ready to be updated: its record, impulse, inverse masses and LDS bodies.
template <int D, typename Real>
struct WgContact {
  typename Vec4<Real>::type g[kRecGroups<D>];
  Real r[3];
  uint32_t ids;  // LDS body of side a (low half) and b (kWgNoBody: a plane)
};
constexpr uint32_t kWgNoBody = 0xFFFFu;

// Orders LDS accesses of the workgroup across colours without waiting for its outstanding
// global accesses: between colours only the velocities in LDS pass from thread to thread (a
// contact's record is read-only and its impulse belongs to one thread).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int D, typename Real>
struct WgSolve {
  using V = typename Vec4<Real>::type;
  using V2 = typename Vec2<Real>::type;
  static constexpr int kBodyV2 = (D == 3) ? 3 : 1;  // LDS vectors per body

  const WgBufs<Real>& W;
  uint32_t C;
  V2* sb;

  __device__ __forceinline__ void load(uint32_t j, WgContact<D, Real>& L) const {
    const V* rec = reinterpret_cast<const V*>(W.rec);
#pragma unroll
    for (int g = 0; g < kRecGroups<D>; ++g) L.g[g] = rec[(size_t)g * C + j];
    L.ids = W.ids[j];
    if constexpr (D == 3) {
      const V r = reinterpret_cast<const V*>(W.r)[j];
      L.r[0] = r.x;
      L.r[1] = r.y;
      L.r[2] = r.z;
    } else {
      const V2 r = reinterpret_cast<const V2*>(W.r)[j];
      L.r[0] = r.x;
      L.r[1] = r.y;
      L.r[2] = 0;
    }
  }

  __device__ __forceinline__ void store_r(uint32_t j, const Real* r) const {
    if constexpr (D == 3) {
      V o = {r[0], r[1], r[2], (Real)0};
      reinterpret_cast<V*>(W.r)[j] = o;
    } else {
      V2 o = {r[0], r[1]};
      reinterpret_cast<V2*>(W.r)[j] = o;
    }
  }

  // Body `id` as the vectors of a body record, with its inverse mass and inertia.
  __device__ __forceinline__ void ld_body(uint32_t id, Real im, Real ii, V& v, V& w) const {
    const V2* b = sb + (size_t)kBodyV2 * id;
    const V2 p = b[0];
    if constexpr (D == 3) {
      const V2 q = b[1], s = b[2];
      v = V{p.x, p.y, q.x, im};
      w = V{q.y, s.x, s.y, ii};
    } else {
      v = V{p.x, p.y, (Real)0, im};
      w = V{0, 0, 0, 0};
    }
  }
  __device__ __forceinline__ void st_body(uint32_t id, const V& v, const V& w) const {
    V2* b = sb + (size_t)kBodyV2 * id;
    b[0] = V2{v.x, v.y};
    if constexpr (D == 3) {
      b[1] = V2{v.z, w.x};
      b[2] = V2{w.y, w.z};
    }
  }

  // One contact of a colour pass (init: apply its impulse). rbest: where its impulse of the
  // previous sweep goes first, or nullptr.
  __device__ __forceinline__ void update(uint32_t j, const WgContact<D, Real>& L, bool init, Real* rbest) const {
    Loaded<D, Real> ld;
    Real im[4];
    unpack_rec<D, Real>(L.g, (L.ids >> 16) != kWgNoBody, ld.R, im);
    ld.r[0] = L.r[0], ld.r[1] = L.r[1], ld.r[2] = L.r[2];
    const uint32_t ia = L.ids & 0xFFFFu, ib = L.ids >> 16;
    const bool hasb = ib != kWgNoBody;
    V b[4];
    ld_body(ia, im[0], im[2], b[0], b[1]);
    ld_body(hasb ? ib : ia, im[1], im[3], b[2], b[3]);
    Real rn[3] = {0, 0, 0};
    update_core<D, Real>(
        ld, init, rbest, 0, 2, [&](size_t i) { return b[i]; }, [&](size_t i, const V& x) { b[i] = x; },
        [&](int d, Real x) { rn[d] = x; });
    st_body(ia, b[0], b[1]);
    if (hasb) st_body(ib, b[2], b[3]);
    if (!init) store_r(j, rn);
  }

  // Squared residual of one contact on the current velocities, in precision T.
  template <typename T>
  __device__ __forceinline__ T residual(const WgContact<D, Real>& L) const {
    Rec<D, Real> R;
    Real im[4];
    unpack_rec<D, Real>(L.g, (L.ids >> 16) != kWgNoBody, R, im);
    const uint32_t ia = L.ids & 0xFFFFu, ib = L.ids >> 16;
    const V z = {0, 0, 0, 0};
    V va, wa, vb = z, wb = z;
    ld_body(ia, im[0], im[2], va, wa);
    if (ib != kWgNoBody) ld_body(ib, im[1], im[3], vb, wb);
    T u[3];
    rel_vel<D, T, Real>(R, va, wa, vb, wb, u);
    const T r[3] = {(T)L.r[0], (T)L.r[1], (T)L.r[2]};
    return fb_err<D, T>((T)R.mu, r, u);
  }
};

// One scene. The solve of k_gs, step for step (phases, stopping rule, best iterate,
// stagnation, skipped evaluations), with every contact updated in the same colour order, so
// the iterates are the same bit for bit.
template <int D, typename Real>
__global__ void __launch_bounds__((kWgThreadsOf<D, Real>)) k_gs_wg(GSArgs<Real> A, WgBufs<Real> W) {
  constexpr uint32_t kWgThreads = kWgThreadsOf<D, Real>;
  using V = typename Vec4<Real>::type;
  using S = WgSolve<D, Real>;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  __shared__ uint32_t off[kMaxColours + 1];
  __shared__ double s_red[kWgThreads / 64];
  __shared__ uint32_t s_nb, s_flag[2];
  const uint32_t tid = threadIdx.x, C = A.C;
  const uint32_t ncol = A.ctr->ncolours;
  S X{W, C, reinterpret_cast<typename S::V2*>(lds)};
  for (uint32_t c = tid; c <= ncol; c += kWgThreads) off[c] = A.coloff[c];
  if (tid == 0) {
    s_nb = 0;
    s_flag[0] = s_flag[1] = 0;
  }
  // The touched bodies numbered 0, 1, ...: every endpoint 2k + side claims its body's word of
  // lmap (all ones between solves), the smallest one takes the next number, loads the body
  // and leaves the number there for the others.
  for (uint32_t k = tid; k < C; k += kWgThreads) {
    atomicMin(&A.lmap[A.c.a[k]], 2 * k);
    if (A.c.b[k] != kNoBody) atomicMin(&A.lmap[A.c.b[k]], 2 * k + 1);
  }
  wait_stores();
  __syncthreads();
  const V* gb = reinterpret_cast<const V*>(A.body);
  constexpr uint32_t kNumbered = 0x80000000u;
  for (uint32_t e = tid; e < 2 * C; e += kWgThreads) {
    const uint32_t sl = (e & 1) ? A.c.b[e >> 1] : A.c.a[e >> 1];
    if (sl == kNoBody) continue;
    if (__hip_atomic_load(&A.lmap[sl], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != e) continue;
    const uint32_t id = atomicAdd(&s_nb, 1u);
    W.slot[id] = sl;
    const V v = gb[(size_t)kBodyVecs<D> * sl];
    V w = {0, 0, 0, 0};
    if (D == 3) w = gb[(size_t)kBodyVecs<D> * sl + 1];
    X.st_body(id, v, w);
    __hip_atomic_store(&A.lmap[sl], kNumbered | id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  wait_stores();
  __syncthreads();
  // packed records
  for (uint32_t k = tid; k < C; k += kWgThreads) {
    Rec<D, Real> R;
    load_rec<D, Real>(A.c, k, R);
    auto number = [&](uint32_t sl) {
      return __hip_atomic_load(&A.lmap[sl], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & ~kNumbered;
    };
    const bool hasb = R.b != kNoBody;
    W.ids[k] = number(R.a) | ((hasb ? number(R.b) : kWgNoBody) << 16);
    pack_rec<D, Real>(R, gb, C, k, reinterpret_cast<V*>(W.rec));
    const Real* rp = A.c.r + 3 * (size_t)k;
    const Real r[3] = {rp[0], rp[1], rp[2]};
    X.store_r(k, r);
  }
  wait_stores();
  __syncthreads();
  for (uint32_t e = tid; e < 2 * C; e += kWgThreads) {
    const uint32_t sl = (e & 1) ? A.c.b[e >> 1] : A.c.a[e >> 1];
    if (sl != kNoBody) __hip_atomic_store(&A.lmap[sl], kNoBody, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // Contact j of a colour belongs to thread (j - off[colour]) mod kWgThreads in every loop
  // (passes of kWgThreads contacts), so its impulse passes through memory within one thread
  // and no barrier waits for it.
  auto own_contacts = [&](auto&& f) {
    for (uint32_t c = 0; c < ncol; ++c)
      for (uint32_t j = off[c] + tid; j < off[c + 1]; j += kWgThreads) f(j);
  };
  // v = v0 + M^-1 H^T r, colour by colour
  auto apply = [&](bool reset) {
    if (reset) {
      for (uint32_t id = tid; id < s_nb; id += kWgThreads) {
        const uint32_t sl = W.slot[id];
        const uint32_t i = A.sid ? A.sid[sl] : sl;
        V v = {(Real)A.v0[(size_t)D * i], (Real)A.v0[(size_t)D * i + 1], (Real)0, (Real)0}, w = {0, 0, 0, 0};
        if (D == 3) {
          v.z = (Real)A.v0[(size_t)D * i + D - 1];
          w = V{(Real)A.w0[3 * (size_t)i], (Real)A.w0[3 * (size_t)i + 1], (Real)A.w0[3 * (size_t)i + 2], (Real)0};
        }
        X.st_body(id, v, w);
      }
      __syncthreads();
    }
    for (uint32_t col = 0; col < ncol; ++col) {
      for (uint32_t j = off[col] + tid; j < off[col + 1]; j += kWgThreads) {
        WgContact<D, Real> L;
        X.load(j, L);
        X.update(j, L, true, nullptr);
      }
      __syncthreads();
    }
  };
  auto contact_residual = [&](const WgContact<D, Real>& L) {
    return A.phase == 1 ? (double)X.template residual<float>(L) : X.template residual<double>(L);
  };
  // max of the residuals; a thread also notes the largest of its contacts at or above
  // `capture` (>= 0), for the check of the sweeps that follow
  uint32_t noted = kNoBody;
  auto evaluate = [&](double capture) {
    double m = 0.0;
    noted = kNoBody;
    for (uint32_t col = 0; col < ncol; ++col) {
#pragma unroll 2
      for (uint32_t j = off[col] + tid; j < off[col + 1]; j += kWgThreads) {
        WgContact<D, Real> L;
        X.load(j, L);
        const double e = contact_residual(L);
        if (capture >= 0.0 && e >= capture && e > m) noted = j;
        m = fmax(m, e);
      }
    }
    m = wave_reduce_max_f64(m);
    if ((tid & 63) == 0) s_red[tid >> 6] = m;
    __syncthreads();
    double out = s_red[0];
    for (int w = 1; w < kWgThreads / 64; ++w) out = fmax(out, s_red[w]);
    __syncthreads();
    return out;
  };

  uint32_t max_iters = A.max_iters;
  if (A.phase == 1) max_iters = max(1u, max_iters - max_iters / 4);
  if (A.phase == 2) max_iters = (A.ctr->sweeps_fp32 < max_iters) ? max_iters - A.ctr->sweeps_fp32 : 0u;
  const bool track_best = A.phase != 1;
  if (A.apply_init) apply(false);
  const double stop = (A.phase == 1) ? 0.5 * A.tol : A.tol;
  const bool subset = A.viol != nullptr;
  // whether the first sweeps of the FP32 phase may go by the stopping value (see WgBufs)
  const bool early = A.phase == 1 && W.skip_early;
  constexpr uint32_t kFullEvery = 256, kSkipUntil = 1024 - kFullEvery;  // as in k_gs
  double err = evaluate(subset ? stop : -1.0);
  uint32_t nev = 1, nskip = 0, nchecks = 0, last_full = 0;
  double best = err, ref = best;
  bool copy_pending = track_best;
  uint32_t ref_it = 0, it = 0;
  if (!(err < stop)) {
    WgContact<D, Real> c0, c1, seen;
    // lowered: the last evaluation found a new best residual below the threshold of its
    // check; while that goes on, the next check would fail as well and is left out
    bool copy = copy_pending, may_skip = false, eval_now = false, lowered = false;
    double th = 0.0;
    auto begin_sweep = [&]() {
      ++it;
      copy = copy_pending;
      copy_pending = false;
      eval_now = A.eval_every > 0 && it % A.eval_every == 0;
      const bool stagnation_due = A.phase == 1 && it - ref_it >= 1024;
      may_skip = subset && eval_now && it - last_full < kFullEvery && !stagnation_due &&
                 !(lowered && last_full + A.eval_every == it);
      th = (early && it < kSkipUntil) ? stop : fmax(stop, best);
    };
    // after the last colour's barrier; true when the solve is over
    auto end_sweep = [&]() {
      if (may_skip) {
        // as violator_check of k_gs: is one of the contacts noted by the last full
        // evaluation still at or above th?
        const uint32_t f = nchecks++ & 1u;
        const bool above = noted != kNoBody && contact_residual(seen) >= th;
        if (__any(above) && (tid & 63) == 0) s_flag[f] = 1u;
        __syncthreads();
        const bool skip = s_flag[f] != 0u;
        if (tid == 0) s_flag[f ^ 1u] = 0u;
        if (skip) {
          ++nskip;
          return false;
        }
      }
      if (eval_now) {
        last_full = it;
        err = evaluate(subset ? fmax(stop, 0.1 * err) : -1.0);
        ++nev;
        lowered = err < th;
        if (err < best) {
          best = err;
          copy_pending = track_best;
        }
        if (err < stop) return true;
        if (A.phase == 1 && it - ref_it >= 1024) {
          if (best > 0.9999 * ref) return true;
          ref = best;
          ref_it = it;
        }
      }
      return false;
    };
    // One pass: kWgThreads contacts of a colour from position pos, held in `use`. The pass
    // after it (of this colour, the next one or the next sweep) is loaded into `fill` first,
    // so its latency passes behind the update and the barrier; two buffers change roles from
    // pass to pass, as a copy between them would wait for the loads.
    uint32_t col = 0, pos = off[0];
    auto pass = [&](const WgContact<D, Real>& use, WgContact<D, Real>& fill) {
      const uint32_t j = pos + tid;
      const bool mine = j < off[col + 1], last = pos + kWgThreads >= off[col + 1];
      const bool sweep_done = last && col + 1 == ncol;
      const uint32_t ncol_ = sweep_done ? 0u : last ? col + 1 : col;
      const uint32_t npos = last ? off[ncol_] : pos + kWgThreads;
      const bool next = npos + tid < off[ncol_ + 1], self = npos == pos;
      if (next && !self) X.load(npos + tid, fill);
      if (mine) X.update(j, use, false, copy ? A.rbest + 3 * (size_t)j : nullptr);
      if (next && self) X.load(npos + tid, fill);  // a single pass: the impulse just stored
      if (last) {
        // the noted contact's record and impulse on their way before the last barrier
        if (sweep_done && may_skip && noted != kNoBody) X.load(noted, seen);
        lds_barrier();
      }
      col = ncol_;
      pos = npos;
      if (!sweep_done) return false;
      if (end_sweep()) return true;
      if (it == max_iters) {
        ++it;
        return true;
      }
      begin_sweep();
      return false;
    };
    if (max_iters > 0) {
      begin_sweep();
      if (off[0] + tid < off[1]) X.load(off[0] + tid, c0);
      while (!pass(c0, c1) && !pass(c1, c0)) {
      }
    } else {
      it = 1;
    }
    __syncthreads();
    if (it > max_iters && track_best && !copy_pending) {
      // the best iterate and its velocities
      own_contacts([&](uint32_t j) {
        const Real r[3] = {A.rbest[3 * (size_t)j], A.rbest[3 * (size_t)j + 1], A.rbest[3 * (size_t)j + 2]};
        X.store_r(j, r);
      });
      apply(true);
    }
    if (it > max_iters) it = max_iters;
  }
  __syncthreads();
  own_contacts([&](uint32_t j) {
    WgContact<D, Real> L;
    X.load(j, L);
    for (int d = 0; d < D; ++d) A.c.r[3 * (size_t)j + d] = L.r[d];
  });
  V* gbw = reinterpret_cast<V*>(A.body);
  for (uint32_t id = tid; id < s_nb; id += kWgThreads) {
    const uint32_t sl = W.slot[id];
    V v, w;
    X.ld_body(id, (Real)0, (Real)0, v, w);
    v.w = gbw[(size_t)kBodyVecs<D> * sl].w;
    gbw[(size_t)kBodyVecs<D> * sl] = v;
    if (D == 3) {
      w.w = gbw[(size_t)kBodyVecs<D> * sl + 1].w;
      gbw[(size_t)kBodyVecs<D> * sl + 1] = w;
    }
  }
  if (tid == 0) {
    if (A.phase == 1) {
      A.ctr->sweeps_fp32 = it;
      A.ctr->error_fp32 = best;
      A.ctr->evals_fp32 = nev;
    }
    A.ctr->sweeps += it;
    A.ctr->error = best;
    A.ctr->evals += nev;
    A.ctr->evals_skipped += nskip;
  }
}

template <int D, typename Real>
size_t wg_lds_bytes(uint32_t nbodies, uint32_t C) {
  // the touched bodies number at most all bodies and at most two per contact
  return (size_t)std::min<uint64_t>(nbodies, 2ull * C) * sizeof(Real) * (D == 3 ? 6 : 2);
}

template <int D, typename Real>
hipError_t launch_gs_wg(const GSArgs<Real>& A, const WgBufs<Real>& W, hipStream_t s) {
  const size_t lds = wg_lds_bytes<D, Real>(A.nbodies, A.C);
  const hipError_t e = hipFuncSetAttribute((const void*)k_gs_wg<D, Real>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)lds);
  if (e != hipSuccess) return e;
  k_gs_wg<D, Real><<<1, kWgThreadsOf<D, Real>, lds, s>>>(A, W);
  return hipGetLastError();
}

template size_t wg_lds_bytes<2, float>(uint32_t, uint32_t);
template size_t wg_lds_bytes<3, float>(uint32_t, uint32_t);
template size_t wg_lds_bytes<2, double>(uint32_t, uint32_t);
template size_t wg_lds_bytes<3, double>(uint32_t, uint32_t);
template hipError_t launch_gs_wg<2, float>(const GSArgs<float>&, const WgBufs<float>&, hipStream_t);
template hipError_t launch_gs_wg<3, float>(const GSArgs<float>&, const WgBufs<float>&, hipStream_t);
template hipError_t launch_gs_wg<2, double>(const GSArgs<double>&, const WgBufs<double>&, hipStream_t);
template hipError_t launch_gs_wg<3, double>(const GSArgs<double>&, const WgBufs<double>&, hipStream_t);

}  // namespace scx
