// scx_solver_flow.hip -- the sweeps of a contact set on many workgroups without barriers
// between the colours: a contact waits only for the contacts before it on its own two bodies.
//
// What bounds the sweeps of a few thousand to a million contacts is neither arithmetic nor
// memory but the exchange of bodies between the colours. With a grid barrier per colour an
// interval costs 8 to 13 us (coherent gathers, the completion of scattered coherent stores,
// the arrival and the slowest workgroup). Here a contact's successors on its two bodies wait
// for it alone, and the way between them is as short as the split of the contacts allows:
//   - A workgroup owns the contacts of a range of bodies that lie together, so most bodies
//     have all their contacts in one workgroup (75 to 85 % of the contacts' bodies on a pile
//     of 262,144 spheres over 256 workgroups). Their velocities stay in its LDS, each with the
//     sweep and colour of its last update, for which the next contact waits.
//   - For the other bodies every contact owns an outbox slot per body: it writes the body's
//     velocities there after its update, in 16-byte pieces that each end in the sweep's tag,
//     and the next contact on that body (the order on a body is the colour order, cyclic over
//     the sweeps) polls that slot until the tag is the one it waits for. A slot whose readers
//     are all on the writer's XCD is stored into its L2 (430 cycles to the next load, which
//     passes the L1 by), others go through to memory (600 to 1,000 cycles).
// No store is waited for, nothing is read that has not been written, and the stores of a wave
// are contiguous. A piece's tag vouches for the three words before it: this rests on an aligned
// 16-byte store of one lane being seen whole by a 16-byte load from any XCD. (It never crosses a
// line, and the memory path moves such a store as one request.)
//
// A hop (wait, solve, store) takes 1,600 cycles through LDS, 2,200 through one XCD's L2 and up to
// 5,000 across XCDs, and a sweep is a chain of about as many hops as there are colours. Measured,
// per FP32 and FP64 sweep (the latter with its residual): 34,176 sphere contacts 18.5 and 36 us
// (with barriers 44.6 and 80), 423,718 sphere contacts 28 and 55 us (59 and 124).
//
// The iterates are those of the colour passes bit for bit: the order of the contacts on
// every body is the colour order, and a contact reads nothing but its own two bodies.
// Progress: the launch is cooperative (every workgroup gets its place once other kernels have
// left it), and the first exchange waits for all of them without a limit. Then a wave takes its
// contacts in colour order, and a contact waits only for contacts of lower colours of its sweep
// or of the sweep before; the order (sweep, colour) has no cycle. A slot is written again only
// by the same contact one sweep later, which follows its reader on the body's cycle. Every wait
// but the first also ends after kFlowPolls looks: the wave then waits no more, its workgroup
// leaves its sweeps when its waves next meet, every wave reports at the kernel's end and the
// step fails.
#pragma clang fp contract(on)

#include "scx_device.h"
#include "scx_internal.h"
#include "scx_sweep.h"

#include <algorithm>

namespace scx {

typedef uint32_t u32x4f __attribute__((ext_vector_type(4)));

constexpr int kFlowThreads = 512;
constexpr size_t kFlowLdsMax = 138 * 1024;  // beside the kernel's static arrays
constexpr int kFlowAux = 16;               // agent scope (SC1)

// 16-byte pieces of a slot: three words of velocity and the tag.
template <int D, typename Real>
constexpr int kSlotPieces = (D == 3) ? (sizeof(Real) == 8 ? 4 : 2) : (sizeof(Real) == 8 ? 2 : 1);

template <int D, typename Real>
struct FlowPort {
  using V = typename Vec4<Real>::type;
  static constexpr int NP = kSlotPieces<D, Real>;
  static constexpr int NR = (D == 3) ? 6 : 2;               // Reals of a body
  static constexpr int NW = NR * (int)sizeof(Real) / 4;     // their words
  __amdgpu_buffer_rsrc_t rs;

  struct Raw {
    u32x4f p[NP];
  };

  // byte offset of a slot; kNowhere: loads read 0, stores go nowhere (beyond the buffer's end)
  static constexpr uint32_t kNowhere = 1u << 31;
  __device__ __forceinline__ static uint32_t at(uint32_t slot) { return slot * (uint32_t)(16 * NP); }
  __device__ __forceinline__ void ld(uint32_t o, Raw& x) const {
#pragma unroll
    for (int i = 0; i < NP; ++i) x.p[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, o + 16u * i, 0, kFlowAux);
  }
  __device__ __forceinline__ static bool is(const Raw& x, uint32_t tag) {
    bool ok = true;
#pragma unroll
    for (int i = 0; i < NP; ++i) ok = ok && x.p[i][3] == tag;
    return ok;
  }
  __device__ __forceinline__ static bool beyond(const Raw& x, uint32_t tag) {
    bool b = false;
#pragma unroll
    for (int i = 0; i < NP; ++i) b = b || (int32_t)(x.p[i][3] - tag) > 0;
    return b;
  }
  __device__ __forceinline__ static void unpack(const Raw& x, Real* r) {
    uint32_t u[3 * NP];
#pragma unroll
    for (int i = 0; i < 3 * NP; ++i) u[i] = x.p[i / 3][i % 3];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      if constexpr (sizeof(Real) == 8)
        r[i] = __longlong_as_double((long long)(((unsigned long long)u[2 * i + 1] << 32) | u[2 * i]));
      else
        r[i] = __uint_as_float(u[i]);
    }
  }
  __device__ __forceinline__ static void pack(const V& v, const V& w, uint32_t tag, Raw& x) {
    Real r[NR];
    if constexpr (D == 3) {
      r[0] = v.x, r[1] = v.y, r[2] = v.z, r[3] = w.x, r[4] = w.y, r[5] = w.z;
    } else {
      r[0] = v.x, r[1] = v.y;
    }
    uint32_t u[3 * NP];
#pragma unroll
    for (int i = 0; i < 3 * NP; ++i) u[i] = 0;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      if constexpr (sizeof(Real) == 8) {
        const unsigned long long b = (unsigned long long)__double_as_longlong(r[i]);
        u[2 * i] = (uint32_t)b;
        u[2 * i + 1] = (uint32_t)(b >> 32);
      } else {
        u[i] = __float_as_uint(r[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < NP; ++i) x.p[i] = u32x4f{u[3 * i], u[3 * i + 1], u[3 * i + 2], tag};
  }
  // Aux 0: every reader is on this XCD, so the store may stay in its L2
  template <int Aux>
  __device__ __forceinline__ void st(uint32_t o, const Raw& x) const {
#pragma unroll
    for (int i = 0; i < NP; ++i) __builtin_amdgcn_raw_buffer_store_b128(x.p[i], rs, o + 16u * i, 0, Aux);
  }
};

// A contact ready to be updated: its record and impulse, and where its bodies come from
// (kFlowHome: LDS entry << 9 | colour of the contact before it << 3; else: slot << 3 | whether
// its own slot of that body is read on this XCD alone (kFlowNear); kFlowWrap: the contact before
// it is one of the sweep before).
template <int D, typename Real>
struct FlowContact {
  typename Vec4<Real>::type g[kRecGroups<D>];
  Real r[3];
  uint32_t from_a, from_b;  // from_b == kNoBody: a plane
  uint32_t scene;           // ensembles
};

// The solve of k_gs, step for step (phases, stopping rule, best iterate, stagnation, skipped
// evaluations). Ens: an ensemble; its scenes share no body, so they are independent parts of
// one graph. A scene is frozen when an evaluation finds it below the tolerance: its contacts
// are neither updated nor evaluated any more, its residual stays in frozen_max.
// All: the LDS holds all contacts of every workgroup (no loads of records from memory, which
// would be waited for behind the stores to the slots).
template <int D, typename Real, bool Ens, bool All>
__global__ void __launch_bounds__(kFlowThreads) k_gs_flow(GSArgs<Real> A, FlowBufs<Real> F) {
  using V = typename Vec4<Real>::type;
  using V2 = typename Vec2<Real>::type;
  using Port = FlowPort<D, Real>;
  using Raw = typename Port::Raw;
  constexpr int kWaves = kFlowThreads / 64;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  __shared__ double s_red[kWaves];
  __shared__ uint32_t s_flag[2], s_skip[2], s_dead;
  __shared__ uint32_t s_beg[kMaxColours + 1], s_rows;
  __shared__ uint32_t s_frozen[Ens ? kFlowMaxScenes / 32 : 1];           // frozen scenes
  __shared__ unsigned long long s_acc[Ens ? kFlowMaxScenes : 1];         // residuals of this workgroup's scenes
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  // The dispatcher deals workgroups to the XCDs round-robin: the workgroups of the first
  // F.xcds XCDs take part, neighbouring ranges of contacts on one XCD.
  const uint32_t per_xcd = gridDim.x / kXcds;
  if (blockIdx.x % kXcds >= F.xcds) return;
  const uint32_t N = flow_places(A.C), G = F.xcds * per_xcd;
  const uint32_t wg = blockIdx.x % kXcds * per_xcd + blockIdx.x / kXcds;
  const uint32_t ncol = A.ctr->ncolours;
  const uint32_t* beg = F.beg + (size_t)wg * (kMaxColours + 1);
  const uint32_t first = beg[0];
  for (uint32_t c = tid; c <= ncol; c += kFlowThreads) s_beg[c] = beg[c];
  if (tid == 0) s_flag[0] = s_flag[1] = s_skip[0] = s_skip[1] = s_dead = 0;
  if (Ens)
    for (uint32_t w = tid; w < kFlowMaxScenes / 32; w += kFlowThreads) s_frozen[w] = 0;
  // The first kept contacts of the workgroup's list (its wide colours) keep their records,
  // impulses and links in LDS.
  const uint32_t kept = F.kept;
  Real* l_body = reinterpret_cast<Real*>(lds);
  uint32_t* l_tag = reinterpret_cast<uint32_t*>(l_body + (size_t)Port::NR * F.home);
  // rows of up to 64 contacts of a colour, in colour order: first place, contacts << 8 | colour
  uint2* l_row = reinterpret_cast<uint2*>(l_tag + F.home);
  V* l_rec = reinterpret_cast<V*>(l_row + F.rows);
  uint2* l_from = reinterpret_cast<uint2*>(l_rec + (size_t)kRecGroups<D> * kept);
  Real* l_r = reinterpret_cast<Real*>(l_from + kept);
  Port P;
  P.rs = __builtin_amdgcn_make_buffer_rsrc(F.slots, (short)0, (int)(4u * N * (uint32_t)(16 * Port::NP)), 0x00020000);
  const __amdgpu_buffer_rsrc_t frs = __builtin_amdgcn_make_buffer_rsrc(F.flags, (short)0, (int)(4u * kFlowMaxBlocks), 0x00020000);
  const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(F.parts, (short)0, (int)(32u * kFlowMaxBlocks), 0x00020000);
  uint32_t tag = F.tag0;  // of the sweep under way
  bool dead = false;      // a wait of this lane ran out
  uint32_t polls = kFlowPolls;  // of a wait for bodies; F.polls during the sweeps
  // Exchanges so far. Their parts lie in two buffers in turn: a workgroup that publishes for
  // exchange n + 2 has seen every part of exchange n + 1, whose owners had read all of n.
  uint32_t nex = 0;
  bool one_l2 = false;    // the workgroups dealt to an XCD are on one XCD

  for (uint32_t i = tid; i < F.home; i += kFlowThreads) l_tag[i] = (tag - 2u) << kFlowColourBits;  // no contact waits for it
  __syncthreads();
  if (tid < 64) {
    const uint32_t n = lane < ncol ? s_beg[lane + 1] - s_beg[lane] : 0u, rows = (n + 63) / 64;
    uint32_t upto = rows;
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)upto, d, 64);
      if ((int)lane >= d) upto += y;
    }
    for (uint32_t r = 0; r < rows; ++r)
      l_row[upto - rows + r] = make_uint2(s_beg[lane] + 64 * r, min(64u, n - 64 * r) << 8 | lane);
    // every wave has as many rows, some of them empty
    const uint32_t all = (uint32_t)__shfl((int)upto, 63, 64), padded = max(1u, (all + kWaves - 1) / kWaves) * kWaves;
    if (all + lane < padded) l_row[all + lane] = make_uint2(first, 0u);
    if (lane == 0) s_rows = padded;
  }
  __syncthreads();
  const uint32_t nrows = s_rows, wave = tid >> 6;
  auto row = [&](uint32_t r) {
    const uint2 d = l_row[r];
    return make_uint2((uint32_t)__builtin_amdgcn_readfirstlane((int)d.x), (uint32_t)__builtin_amdgcn_readfirstlane((int)d.y));
  };
  // the contact at place j
  auto load = [&](uint32_t j, FlowContact<D, Real>& L) __attribute__((always_inline)) {
    const uint32_t i = j - first;
    if (Ens) L.scene = F.scene[j];
    if (All || i < kept) {
#pragma unroll
      for (int g = 0; g < kRecGroups<D>; ++g) L.g[g] = l_rec[(size_t)g * kept + i];
      const uint2 f = l_from[i];
      L.from_a = f.x;
      L.from_b = f.y;
#pragma unroll
      for (int d = 0; d < D; ++d) L.r[d] = l_r[(size_t)d * kept + i];
      if (D == 2) L.r[2] = 0;
      return;
    }
    const V* rec = reinterpret_cast<const V*>(F.rec);
#pragma unroll
    for (int g = 0; g < kRecGroups<D>; ++g) L.g[g] = rec[(size_t)g * N + j];
    const uint2 f = reinterpret_cast<const uint2*>(F.from)[j];
    L.from_a = f.x;
    L.from_b = f.y;
    if constexpr (D == 3) {
      const V r = reinterpret_cast<const V*>(F.r)[j];
      L.r[0] = r.x, L.r[1] = r.y, L.r[2] = r.z;
    } else {
      const V2 r = reinterpret_cast<const V2*>(F.r)[j];
      L.r[0] = r.x, L.r[1] = r.y, L.r[2] = 0;
    }
  };
  auto store_r = [&](uint32_t j, const Real* r) {
    const uint32_t i = j - first;
    if (All || i < kept) {
#pragma unroll
      for (int d = 0; d < D; ++d) l_r[(size_t)d * kept + i] = r[d];
    } else if constexpr (D == 3) {
      reinterpret_cast<V*>(F.r)[j] = V{r[0], r[1], r[2], (Real)0};
    } else {
      reinterpret_cast<V2*>(F.r)[j] = V2{r[0], r[1]};
    }
  };
  // the slot that the contact at place j writes for a body: near ones after the far ones
  auto own_slot = [&](uint32_t j, uint32_t side, uint32_t from) {
    return j + (side ? N : 0u) + ((from & kFlowNear) ? 2u * N : 0u);
  };
  // Bodies in LDS. A wave's LDS accesses are carried out in their order: a writer stores the
  // velocities before the tag, a reader loads the tag before the velocities. The last 64
  // entries are nobody's: a lane with a body in a slot reads and writes its own of them, so that
  // a wave goes through with few branches (a contact's successors wait for each instruction
  // between).
  const uint32_t nobody = F.home - 64 + lane;
  auto home_of = [&](uint32_t word, bool home) { return home ? word >> (3 + kFlowColourBits) : nobody; };
  auto home_tag = [&](uint32_t word, uint32_t t) { return t << kFlowColourBits | ((word >> 3) & (kMaxColours - 1)); };
  auto home_ld = [&](uint32_t e, Real* x) __attribute__((always_inline)) {
    const V2* p = reinterpret_cast<const V2*>(l_body + (size_t)Port::NR * e);
#pragma unroll
    for (int i = 0; i < Port::NR / 2; ++i) {
      const V2 y = p[i];
      x[2 * i] = y.x, x[2 * i + 1] = y.y;
    }
  };
  auto home_st = [&](uint32_t e, const V& v, const V& w) __attribute__((always_inline)) {
    V2* p = reinterpret_cast<V2*>(l_body + (size_t)Port::NR * e);
    p[0] = V2{v.x, v.y};
    if constexpr (D == 3) {
      p[1] = V2{v.z, w.x};
      p[2] = V2{w.y, w.z};
    }
  };
  auto as_body = [&](const Real* x, Real im, Real ii, V& v, V& w) __attribute__((always_inline)) {
    if constexpr (D == 3) {
      v = V{x[0], x[1], x[2], im};
      w = V{x[3], x[4], x[5], ii};
    } else {
      v = V{x[0], x[1], (Real)0, im};
      w = V{0, 0, 0, 0};
    }
  };
  auto is_home = [&](uint32_t word, bool has) { return has && (word & kFlowHome); };
  // (Waves of equal priority share the issue slots, also those of a wave that only polls: with
  // the lower priority of a wait whole solves take 2 to 5 % less.)
  // Waits for two bodies under the tags ta and tb (b only with hasb). check: gives up (false)
  // when a body in a slot has already moved on to a later sweep (one in LDS moves on with this
  // workgroup only).
  auto gather = [&](uint32_t wa, uint32_t ta, bool hasb, uint32_t wb, uint32_t tb, bool check, Real* xa, Real* xb) __attribute__((always_inline)) {
    const bool ha = is_home(wa, true), hb = is_home(wb, hasb), sa = !ha, sb = hasb && !hb;
    const uint32_t ia = home_of(wa, ha), ib = home_of(wb, hb), ea = home_tag(wa, ta), eb = home_tag(wb, tb);
    const uint32_t oa = sa ? Port::at(wa >> 3) : Port::kNowhere, ob = sb ? Port::at(wb >> 3) : Port::kNowhere;
    const bool slots = __any(sa || sb);  // (a wave without does not wait for its stores to slots)
    bool ok = false, late = false;
    __builtin_amdgcn_s_setprio(0);  // a wave that waits gives way to its SIMD's other wave
    for (uint32_t n = 0; !ok && !late && !dead;) {
      asm volatile("" ::: "memory");  // each look reads memory again
      Raw ra, rb;
      if (slots) {
        P.ld(oa, ra);
        P.ld(ob, rb);
      }
      const uint32_t la = l_tag[ia], lb = l_tag[ib];
      asm volatile("" ::: "memory");
      home_ld(ia, xa);
      home_ld(ib, xb);
      bool oka = la == ea, okb = lb == eb;
      if (slots) {
        Real ya[Port::NR], yb[Port::NR];
        Port::unpack(ra, ya);
        Port::unpack(rb, yb);
#pragma unroll
        for (int i = 0; i < Port::NR; ++i) {
          xa[i] = sa ? ya[i] : xa[i];
          xb[i] = sb ? yb[i] : xb[i];
        }
        oka = sa ? Port::is(ra, ta) : oka;
        okb = sb ? Port::is(rb, tb) : okb;
        if (check) late = (sa && Port::beyond(ra, ta)) || (sb && Port::beyond(rb, tb));
      }
      ok = oka && (okb || !hasb);
      if (!ok && ++n >= polls) dead = true;
    }
    __builtin_amdgcn_s_setprio(3);
    return ok;
  };
  // Stores the bodies of the contact at place j, of colour col, under the sweep's tag.
  auto scatter = [&](uint32_t j, uint32_t col, uint32_t wa, bool hasa, uint32_t wb, bool hasb, const V* b) __attribute__((always_inline)) {
    const bool ha = is_home(wa, hasa), hb = is_home(wb, hasb), sa = hasa && !ha, sb = hasb && !hb;
    const uint32_t ia = home_of(wa, ha), ib = home_of(wb, hb);
    home_st(ia, b[0], b[1]);
    home_st(ib, b[2], b[3]);
    asm volatile("" ::: "memory");
    l_tag[ia] = tag << kFlowColourBits | col;
    l_tag[ib] = tag << kFlowColourBits | col;
    if (__any(sa || sb)) {
      Raw ra, rb;
      Port::pack(b[0], b[1], tag, ra);
      Port::pack(b[2], b[3], tag, rb);
      const bool na = one_l2 && (wa & kFlowNear), nb = one_l2 && (wb & kFlowNear);
      const uint32_t oa = Port::at(own_slot(j, 0, wa)), ob = Port::at(own_slot(j, 1, wb));
      if (__any((sa && na) || (sb && nb))) {
        P.template st<0>(sa && na ? oa : Port::kNowhere, ra);
        P.template st<0>(sb && nb ? ob : Port::kNowhere, rb);
      }
      if (__any((sa && !na) || (sb && !nb))) {
        P.template st<kFlowAux>(sa && !na ? oa : Port::kNowhere, ra);
        P.template st<kFlowAux>(sb && !nb ? ob : Port::kNowhere, rb);
      }
    }
  };
  auto update = [&](uint32_t j, uint32_t col, const FlowContact<D, Real>& L, bool init, Real* rbest) __attribute__((always_inline)) {
    const bool hasb = L.from_b != kNoBody;
    Loaded<D, Real> ld;
    Real im[4];
    unpack_rec<D, Real>(L.g, hasb, ld.R, im);
    ld.r[0] = L.r[0], ld.r[1] = L.r[1], ld.r[2] = L.r[2];
    Real xa[Port::NR], xb[Port::NR];
    (void)gather(L.from_a, tag - (L.from_a & kFlowWrap), hasb, L.from_b, tag - (L.from_b & kFlowWrap), false, xa, xb);
    V b[4];
    as_body(xa, im[0], im[2], b[0], b[1]);
    as_body(xb, im[1], im[3], b[2], b[3]);
    Real rn[3] = {0, 0, 0};
    update_core<D, Real>(
        ld, init, rbest, 0, 2, [&](size_t i) { return b[i]; }, [&](size_t i, const V& x) { b[i] = x; },
        [&](int d, Real x) { rn[d] = x; });
    scatter(j, col, L.from_a, true, L.from_b, hasb, b);
    if (!init) store_r(j, rn);
  };
  // squared residual of contact j on the bodies' final velocities of this sweep; false when a
  // body has already moved on to a later sweep (only in the check of a noted contact)
  auto residual = [&](const FlowContact<D, Real>& L, uint2 fin, bool check, double& e) __attribute__((always_inline)) {
    const bool hasb = fin.y != kNoBody;
    Real xa[Port::NR], xb[Port::NR];
    if (!gather(fin.x, tag, hasb, fin.y, tag, check, xa, xb)) return false;
    Rec<D, Real> R;
    Real im[4];
    unpack_rec<D, Real>(L.g, hasb, R, im);
    const V z = {0, 0, 0, 0};
    V va, wa, vb = z, wb = z;
    as_body(xa, im[0], im[2], va, wa);
    if (hasb) as_body(xb, im[1], im[3], vb, wb);
    if (A.phase == 1) {
      float u[3];
      rel_vel<D, float, Real>(R, va, wa, vb, wb, u);
      const float r[3] = {(float)L.r[0], (float)L.r[1], (float)L.r[2]};
      e = (double)fb_err<D, float>((float)R.mu, r, u);
    } else {
      double u[3];
      rel_vel<D, double, Real>(R, va, wa, vb, wb, u);
      const double r[3] = {(double)L.r[0], (double)L.r[1], (double)L.r[2]};
      e = fb_err<D, double>((double)R.mu, r, u);
    }
    return true;
  };
  auto frozen = [&](const FlowContact<D, Real>& L) {
    return Ens && ((s_frozen[L.scene >> 5] >> (L.scene & 31)) & 1u) != 0;
  };
  // every contact of this wave, in colour order: place j, colour c
  auto for_each = [&](auto&& f) {
    for (uint32_t r = wave; r < nrows; r += kWaves) {
      const uint2 d = row(r);
      if (lane < d.y >> 8) f(d.x + lane, d.y & 0xFFu);
    }
  };
  // whether the contact (place j, colour c) is the last on its body of a side
  auto is_last = [&](uint32_t j, uint32_t c, uint32_t side, uint32_t from, uint32_t fin) {
    if (fin == kNoBody) return false;
    if (fin & kFlowHome) return ((fin >> 3) & (kMaxColours - 1)) == c;
    return fin >> 3 == own_slot(j, side, from);
  };
  // the bodies' start velocities, as their last contacts of the sweep before leave them
  auto start_bodies = [&](bool reset) {
    for_each([&](uint32_t j, uint32_t c) {
      const uint2 fin = reinterpret_cast<const uint2*>(F.fin)[j], fr = reinterpret_cast<const uint2*>(F.from)[j];
      const uint32_t k = F.who[j];
      for (int side = 0; side < 2; ++side) {
        const uint32_t word = side ? fr.y : fr.x;
        if (!is_last(j, c, side, word, side ? fin.y : fin.x)) continue;
        const uint32_t sl = side ? A.c.b[k] : A.c.a[k];
        V v, w = {0, 0, 0, 0};
        if (reset) {
          const uint32_t i = A.sid ? A.sid[sl] : sl;
          v = V{(Real)A.v0[(size_t)D * i], (Real)A.v0[(size_t)D * i + 1], (Real)0, (Real)0};
          if (D == 3) {
            v.z = (Real)A.v0[(size_t)D * i + D - 1];
            w = V{(Real)A.w0[3 * (size_t)i], (Real)A.w0[3 * (size_t)i + 1], (Real)A.w0[3 * (size_t)i + 2], (Real)0};
          }
        } else {
          const V* rec = reinterpret_cast<const V*>(A.body) + (size_t)kBodyVecs<D> * sl;
          v = rec[0];
          if (D == 3) w = rec[1];
        }
        const V b[4] = {v, w, v, w};
        scatter(j, c, word, side == 0, word, side == 1, b);
      }
    });
  };
  auto apply = [&]() {
    for_each([&](uint32_t j, uint32_t c) {
      FlowContact<D, Real> L;
      load(j, L);
      update(j, c, L, true, nullptr);
    });
  };
  // the largest of the workgroups' values published under the current tag, the same in every
  // thread; every workgroup has arrived when it returns
  auto exchange = [&](double m) __attribute__((always_inline)) {
    m = wave_reduce_max_f64(m);
    if (lane == 0) s_red[tid >> 6] = m;
    if (__any(dead) && lane == 0) s_dead = 1;
    if (Ens) wait_stores();  // the scenes' residuals are in memory before the workgroup arrives
    __syncthreads();
    if (tid < 64) {
      double b = lane < kWaves ? s_red[lane] : 0.0;
      b = wave_reduce_max_f64(b);
      if (lane == 0) {
        const unsigned long long u = (unsigned long long)__double_as_longlong(b);
        const u32x4f x = {(uint32_t)u, (uint32_t)(u >> 32), 0u, tag};
        __builtin_amdgcn_raw_buffer_store_b128(x, prs, (nex & 1u) * 16u * kFlowMaxBlocks + wg * 16u, 0, kFlowAux);
      }
      double all = 0.0;
      for (uint32_t g = lane; g < G; g += 64) {
        bool ok = false;
        for (uint32_t n = 0; !ok && !dead; ++n) {
          asm volatile("" ::: "memory");
          const u32x4f x =
              __builtin_amdgcn_raw_buffer_load_b128(prs, (nex & 1u) * 16u * kFlowMaxBlocks + g * 16u, 0, kFlowAux);
          ok = x[3] == tag;
          if (ok) all = fmax(all, __longlong_as_double((long long)(((unsigned long long)x[1] << 32) | x[0])));
          if (n >= kFlowPolls) dead = true;
        }
      }
      all = wave_reduce_max_f64(all);
      if (__any(dead) && lane == 0) s_dead = 1;
      if (lane == 0) s_red[0] = all;
    }
    __syncthreads();
    const double out = s_red[0];
    ++nex;
    __syncthreads();
    return out;
  };
  // the largest residual of the sweep just done over all workgroups, the same in every thread;
  // a thread also notes the largest of its contacts at or above `capture` (>= 0)
  uint32_t noted = kNoBody;
  uint2 noted_fin = make_uint2(0, 0);
  const double stop = (A.phase == 1) ? 0.5 * A.tol : A.tol;
  uint32_t nev = 0;  // evaluations
  double frozen_max = 0.0;
  auto evaluate = [&](double capture, uint32_t sweeps) __attribute__((always_inline)) {
    double m = 0.0;
    noted = kNoBody;
    // Ensembles: three buffers of the scenes' residuals in turn. This evaluation's was cleared
    // during the last one; the next one's, which every workgroup is through with since it
    // arrived at the last exchange, is cleared now.
    unsigned long long* acc = A.scene_acc + (size_t)(nev % 3) * A.nscenes;
    if (Ens) {
      unsigned long long* clear = A.scene_acc + (size_t)((nev + 1) % 3) * A.nscenes;
      for (uint32_t sc = wg * kFlowThreads + tid; sc < A.nscenes; sc += G * kFlowThreads)
        __hip_atomic_store(clear + sc, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      for (uint32_t sc = tid; sc < A.nscenes; sc += kFlowThreads) s_acc[sc] = 0ull;
      __syncthreads();
    }
    for_each([&](uint32_t j, uint32_t) {
      FlowContact<D, Real> L;
      load(j, L);
      if (frozen(L)) return;
      const uint2 fin = reinterpret_cast<const uint2*>(F.fin)[j];
      double e = 0.0;
      residual(L, fin, false, e);
      if (Ens && e > 0.0) atomicMax(s_acc + L.scene, (unsigned long long)__double_as_longlong(e));
      if (capture >= 0.0 && e >= capture && e > m) {
        noted = j;
        noted_fin = fin;
      }
      m = fmax(m, e);
    });
    if (Ens) {
      __syncthreads();
      for (uint32_t sc = tid; sc < A.nscenes; sc += kFlowThreads)
        if (s_acc[sc] != 0ull) atomicMax(acc + sc, s_acc[sc]);
    }
    double out = exchange(m);
    ++nev;
    if (Ens) {
      out = fmax(out, frozen_max);
      auto of_scene = [&](uint32_t sc) {
        return __longlong_as_double(
            (long long)__hip_atomic_load(acc + sc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      };
      double fm = 0.0;
      for (uint32_t b0 = 0; b0 < A.nscenes; b0 += kFlowThreads) {
        const uint32_t sc = b0 + tid;
        const uint32_t w = sc >> 5;
        const bool was = sc < A.nscenes && ((s_frozen[w] >> (sc & 31)) & 1u) != 0;
        const double es = sc < A.nscenes && !was ? of_scene(sc) : 0.0;
        const bool now_f = sc < A.nscenes && !was && es < stop;
        if (now_f) fm = fmax(fm, es);
        const unsigned long long bal = __ballot(now_f || was);
        if ((sc & 31) == 0 && sc < A.nscenes) s_frozen[w] = (uint32_t)(bal >> (lane & 32));
        // one thread of the grid keeps the scene's sweep count
        if (sc < A.nscenes && !was && sc % (G * kFlowThreads) == wg * kFlowThreads + tid % kFlowThreads) {
          if (now_f) {
            if (A.scene_sweeps[sc] == kNoBody) A.scene_sweeps[sc] = sweeps;
          } else if (A.phase == 2) {
            A.scene_sweeps[sc] = kNoBody;  // an FP32 estimate below the tolerance was not confirmed
          }
        }
      }
      fm = wave_reduce_max_f64(fm);
      if (lane == 0) s_red[tid >> 6] = fm;
      __syncthreads();
      for (int w = 0; w < kWaves; ++w) frozen_max = fmax(frozen_max, s_red[w]);
      __syncthreads();
    }
    return out;
  };

  uint32_t max_iters = A.max_iters;
  if (A.phase == 1) max_iters = max(1u, max_iters - max_iters / 4);
  if (A.phase == 2) max_iters = (A.ctr->sweeps_fp32 < max_iters) ? max_iters - A.ctr->sweeps_fp32 : 0u;
  const bool track_best = A.phase != 1;
  for_each([&](uint32_t j, uint32_t) {
    const uint32_t i = j - first;
    if (i >= kept) return;
    const V* rec = reinterpret_cast<const V*>(F.rec);
#pragma unroll
    for (int g = 0; g < kRecGroups<D>; ++g) l_rec[(size_t)g * kept + i] = rec[(size_t)g * N + j];
    l_from[i] = reinterpret_cast<const uint2*>(F.from)[j];
#pragma unroll
    for (int d = 0; d < D; ++d) l_r[(size_t)d * kept + i] = F.r[(size_t)(D == 3 ? 4 : 2) * j + d];
  });
  {
    // Every workgroup's XCD, published and read like the residuals. This is also the wait for the
    // workgroups to become resident: one needs nearly a whole CU's LDS, and a kernel of another
    // context may hold that for as long as it runs, so it has no limit.
    if (tid < 64) {
      const uint32_t xcc = __builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11));  // XCC_ID
      const u32x4f mine = {xcc, 0u, 0u, tag};
      if (lane == 0) __builtin_amdgcn_raw_buffer_store_b128(mine, prs, wg * 16u, 0, kFlowAux);
      bool same = true;
      for (uint32_t g = lane; g < G; g += 64) {
        for (bool ok = false; !ok;) {
          asm volatile("" ::: "memory");
          const u32x4f x = __builtin_amdgcn_raw_buffer_load_b128(prs, g * 16u, 0, kFlowAux);
          const u32x4f y = __builtin_amdgcn_raw_buffer_load_b128(prs, g / per_xcd * per_xcd * 16u, 0, kFlowAux);
          ok = x[3] == tag && y[3] == tag;
          same = same && (!ok || x[0] == y[0]);
          if (!ok) __builtin_amdgcn_s_sleep(1);
        }
      }
      const bool all = __all(same);
      if (lane == 0) s_skip[0] = all ? 1u : 0u;
    }
    __syncthreads();
    one_l2 = s_skip[0] != 0u;
    ++nex;
    ++tag;
  }
  start_bodies(false);
  if (A.apply_init) {
    ++tag;
    apply();
  }
  const uint32_t base = (A.phase == 2) ? A.ctr->sweeps_fp32 : 0u;
  const bool subset = A.viol != nullptr;
  const bool early = A.phase == 1 && F.skip_early;
  constexpr uint32_t kFullEvery = 256, kSkipUntil = 1024 - kFullEvery;  // as in k_gs
  double err = evaluate(subset ? stop : -1.0, base);
  uint32_t nskip = 0, nchecks = 0, last_full = 0;
  double best = err, ref = best;
  bool copy_pending = track_best;
  uint32_t ref_it = 0, it = 0;
  if (!(err < stop) && max_iters > 0) {
    FlowContact<D, Real> c0, c1;
    // lowered: the last evaluation found a new best residual below the threshold of its
    // check; while that goes on, the next check would fail as well and is left out
    bool copy = copy_pending, may_skip = false, eval_now = false, lowered = false;
    double th = 0.0;
    auto begin_sweep = [&]() {
      ++it;
      ++tag;
      copy = copy_pending;
      copy_pending = false;
      eval_now = A.eval_every > 0 && it % A.eval_every == 0;
      const bool stagnation_due = A.phase == 1 && it - ref_it >= 1024;
      may_skip = subset && eval_now && it - last_full < kFullEvery && !stagnation_due &&
                 !(lowered && last_full + A.eval_every == it);
      th = (early && it < kSkipUntil) ? stop : fmax(stop, best);
    };
    // true when the solve is over
    auto end_sweep = [&]() __attribute__((always_inline)) {
      if (may_skip) {
        // Is one of the contacts noted by the last full evaluation still at or above th? A
        // workgroup that has one goes on at once; the others go on when they see its flag (or
        // that it is past this sweep). Only when every workgroup has none is the sweep
        // evaluated, and then none has gone on. A noted contact whose body has moved on
        // means that another workgroup went on, so this one's answer no longer counts.
        const uint32_t f = nchecks++ & 1u;
        bool above = false;
        if (noted != kNoBody) {
          FlowContact<D, Real> L;
          load(noted, L);
          double e = 0.0;
          above = residual(L, noted_fin, true, e) && e >= th;
        }
        if (__any(above) && lane == 0) s_flag[f] = 1u;
        if (__any(dead) && lane == 0) s_dead = 1u;
        __syncthreads();
        if (tid < 64) {
          bool skip = s_flag[f] != 0u;
          if (lane == 0)
            __builtin_amdgcn_raw_buffer_store_b32(2u * tag + (skip ? 1u : 0u), frs, wg * 4u, 0, kFlowAux);
          bool all = skip;
          for (uint32_t n = 0; !all && !dead; ++n) {
            asm volatile("" ::: "memory");
            const uint32_t g = 4 * lane;
            int32_t d[4] = {0, 0, 0, 0};
            if (g < G) {
              const u32x4f x = __builtin_amdgcn_raw_buffer_load_b128(frs, 4u * g, 0, kFlowAux);
#pragma unroll
              for (int i = 0; i < 4; ++i) d[i] = g + i < G ? (int32_t)(x[i] - 2u * tag) : 0;
            }
            bool any = false, here = true;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              any = any || d[i] > 0;
              here = here && d[i] >= 0;
            }
            skip = __any(any);
            all = skip || __all(here);
            if (n >= kFlowPolls) dead = true;
          }
          if (lane == 0) {
            s_skip[f] = skip ? 1u : 0u;
            if (dead) s_dead = 1u;
            s_flag[f ^ 1u] = 0u;
          }
        }
        __syncthreads();
        if (s_dead) return true;
        if (s_skip[f]) {
          ++nskip;
          return false;
        }
      }
      if (eval_now) {
        last_full = it;
        err = evaluate(subset ? fmax(stop, 0.1 * err) : -1.0, base + it);
        if (s_dead) return true;
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
    // One pass: a row, held in `use`; the records of the wave's next row are loaded into `fill`
    // first, behind the wait and the update. The rows are dealt to the waves in turn, so the
    // late colours, of a row or less, don't all fall to one wave.
    uint32_t r = wave;
    uint2 cur = row(wave);
    auto pass = [&](const FlowContact<D, Real>& use, FlowContact<D, Real>& fill) __attribute__((always_inline)) {
      dead = __any(dead);
      const bool sweep_done = r + kWaves >= nrows, self = nrows == kWaves;
      r = sweep_done ? wave : r + kWaves;
      const uint2 nxt = row(r);
      const uint32_t j = cur.x + lane;
      const bool next = lane < nxt.y >> 8;
      if (next && !self) load(nxt.x + lane, fill);
      if (lane < cur.y >> 8) {
        Real* rb = copy ? A.rbest + 3 * (size_t)j : nullptr;
        if (!frozen(use)) {
          update(j, cur.y & 0xFFu, use, false, rb);
        } else if (rb) {
          for (int d = 0; d < 3; ++d) rb[d] = use.r[d];
        }
      }
      if (next && self) load(nxt.x + lane, fill);  // a single row: the impulse just stored
      cur = nxt;
      return sweep_done;
    };
    auto sweep_over = [&]() __attribute__((always_inline)) {
      if (end_sweep()) return true;
      if (it == max_iters) {
        ++it;
        return true;
      }
      begin_sweep();
      return false;
    };
    begin_sweep();
    polls = F.polls;
    if (lane < cur.y >> 8) load(cur.x + lane, c0);
    if constexpr (Ens) {  // one copy of the larger evaluation
      for (bool odd = false;; odd = !odd)
        if ((odd ? pass(c1, c0) : pass(c0, c1)) && sweep_over()) break;
    } else {
      for (;;) {
        if (pass(c0, c1) && sweep_over()) break;
        if (pass(c1, c0) && sweep_over()) break;
      }
    }
    if (it > max_iters) {
      it = max_iters;
      if (track_best && !copy_pending) {
        // the best iterate and its velocities: v0, then its impulses in colour order, once
        // every workgroup is through with the last sweep's slots
        for_each([&](uint32_t j, uint32_t) {
          if (Ens && ((s_frozen[F.scene[j] >> 5] >> (F.scene[j] & 31)) & 1u)) return;  // keeps its impulses
          const Real r[3] = {A.rbest[3 * (size_t)j], A.rbest[3 * (size_t)j + 1], A.rbest[3 * (size_t)j + 2]};
          store_r(j, r);
        });
        ++tag;
        (void)exchange(0.0);
        ++tag;
        start_bodies(true);
        ++tag;
        apply();
      }
    }
  }
  wait_stores();
  // impulses, and the velocities of the bodies whose last contact is here
  for_each([&](uint32_t j, uint32_t c) {
    FlowContact<D, Real> L;
    load(j, L);
    const uint32_t k = F.who[j];
    for (int d = 0; d < D; ++d) A.c.r[3 * (size_t)k + d] = L.r[d];
    const uint2 fin = reinterpret_cast<const uint2*>(F.fin)[j];
    for (int side = 0; side < 2; ++side) {
      const uint32_t word = side ? L.from_b : L.from_a;
      if (!is_last(j, c, side, word, side ? fin.y : fin.x)) continue;
      const uint32_t sl = side ? A.c.b[k] : A.c.a[k];
      Real x[Port::NR];
      if (word & kFlowHome) {
        home_ld(home_of(word, true), x);
      } else {
        Raw raw;
        P.ld(Port::at(own_slot(j, side, word)), raw);
        Port::unpack(raw, x);
      }
      V v, w;
      V* rec = reinterpret_cast<V*>(A.body) + (size_t)kBodyVecs<D> * sl;
      as_body(x, rec[0].w, (D == 3) ? rec[D == 3].w : (Real)0, v, w);
      rec[0] = v;
      if (D == 3) rec[1] = w;
    }
  });
  // (a wait may have run out after the waves last met)
  const bool ran_out = __any(dead) || s_dead;
  if (lane == 0 && ran_out) atomicOr(&A.ctr->wait_ran_out, 1u);
  if (wg == 0 && tid == 0) {
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

// ---------------------------------------------------------------------------
// Links of the contact graph: per body its contacts in colour order (a body has at most one
// contact of a colour, so the set of its colours orders them).
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t colour_of(const uint32_t* off, uint32_t ncol, uint32_t k) {
  uint32_t lo = 0, hi = ncol - 1;  // the last colour that starts at or before k
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (off[mid] <= k) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// The workgroup of contact k (colour c): with first, the number of contacts before those of
// each first body in the order of the bodies (neighbours are near each other in it, and the
// contacts of a colour are sorted by it), the contacts of an equal share of them; else equal
// shares of each colour. Either way it does not fall within a colour.
__device__ __forceinline__ uint32_t flow_owner(uint32_t k, uint32_t a, uint32_t C, uint32_t o0, uint32_t o1,
                                               const uint32_t* first, uint32_t G) {
  if (first) return (uint32_t)((uint64_t)first[a] * G / C);
  return (uint32_t)((((uint64_t)(k - o0) + 1) * G - 1) / (o1 - o0));
}

__global__ void __launch_bounds__(kBlock) k_flow_colours(uint32_t C, const uint32_t* __restrict__ ca,
                                                         const uint32_t* __restrict__ cb,
                                                         const uint32_t* __restrict__ coloff,
                                                         const StepCounters* __restrict__ ctr,
                                                         const uint32_t* __restrict__ first, uint32_t G,
                                                         unsigned long long* __restrict__ mask,
                                                         uint32_t* __restrict__ own) {
  __shared__ uint32_t off[kMaxColours + 1];
  const uint32_t ncol = ctr->ncolours;
  for (uint32_t c = threadIdx.x; c <= ncol; c += kBlock) off[c] = coloff[c];
  __syncthreads();
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= C) return;
  const uint32_t c = colour_of(off, ncol, k);
  const unsigned long long m = 1ull << c;
  atomicOr(&mask[ca[k]], m);
  if (cb[k] != kNoBody) atomicOr(&mask[cb[k]], m);
  own[k] = flow_owner(k, ca[k], C, off[c], off[c + 1], first, G);
}

// lo[w][c]: the first contact of colour c that belongs to workgroup w or a later one.
__global__ void __launch_bounds__(kBlock) k_flow_ranges(uint32_t G, const uint32_t* __restrict__ coloff,
                                                        const StepCounters* __restrict__ ctr,
                                                        const uint32_t* __restrict__ own, uint32_t* __restrict__ lo) {
  const uint32_t c = blockIdx.x;
  if (c >= ctr->ncolours) return;
  const uint32_t o0 = coloff[c], o1 = coloff[c + 1];
  for (uint32_t w = threadIdx.x; w <= G; w += kBlock) {
    uint32_t a = o0, b = o1;
    while (a < b) {
      const uint32_t mid = (a + b) >> 1;
      if (own[mid] < w) a = mid + 1;
      else b = mid;
    }
    lo[(size_t)w * (kMaxColours + 1) + c] = a;
  }
}

// beg[w][c]: the place of workgroup w's first contact of colour c (c = ncolours: the end).
// Workgroup after workgroup, a line's worth of places free between the XCDs.
__global__ void __launch_bounds__(kMaxColours) k_flow_places(uint32_t per_xcd, const uint32_t* __restrict__ coloff,
                                                             const StepCounters* __restrict__ ctr,
                                                             const uint32_t* __restrict__ lo,
                                                             uint32_t* __restrict__ beg,
                                                             uint32_t* __restrict__ homes) {
  static_assert(kMaxColours == 64, "one wave, a lane per colour");
  const uint32_t w = blockIdx.x, c = threadIdx.x, ncol = ctr->ncolours;
  const uint32_t* l = lo + (size_t)w * (kMaxColours + 1);
  uint32_t before = c < ncol ? l[c] - coloff[c] : 0u;  // contacts of earlier workgroups
  const uint32_t mine = c < ncol ? l[kMaxColours + 1 + c] - l[c] : 0u;
  uint32_t upto = mine;
  for (int d = 1; d < 64; d <<= 1) {
    before += (uint32_t)__shfl_xor((int)before, d, 64);
    const uint32_t y = (uint32_t)__shfl_up((int)upto, d, 64);
    if ((int)c >= d) upto += y;
  }
  uint32_t* o = beg + (size_t)w * (kMaxColours + 1);
  const uint32_t base = before + w / per_xcd * kFlowLine;
  o[c] = base + upto - mine;
  if (c == 63) o[64] = base + upto;
  if (c == 0) homes[w] = 0;
}

// Start of each body's entries in the table (any order of the bodies); mask[n] counts them.
__global__ void __launch_bounds__(kBlock) k_flow_offsets(uint32_t n, unsigned long long* __restrict__ mask,
                                                         uint32_t* __restrict__ start) {
  __shared__ uint32_t s_base;
  const uint32_t b = blockIdx.x * kBlock + threadIdx.x;
  const uint32_t deg = b < n ? (uint32_t)__popcll(mask[b]) : 0u;
  uint32_t total;
  const uint32_t before = block_exclusive_scan_u32(deg, &total);
  if (threadIdx.x == 0) s_base = total ? atomicAdd(reinterpret_cast<uint32_t*>(mask + n), total) : 0u;
  __syncthreads();
  if (b < n) start[b] = s_base + before;
}

// The body's contact of each of its colours (contact, its side in the top bit), and the
// contacts' places.
__global__ void __launch_bounds__(kBlock) k_flow_table(uint32_t C, const uint32_t* __restrict__ ca,
                                                       const uint32_t* __restrict__ cb,
                                                       const uint32_t* __restrict__ coloff,
                                                       const StepCounters* __restrict__ ctr,
                                                       const unsigned long long* __restrict__ mask,
                                                       const uint32_t* __restrict__ start,
                                                       const uint32_t* __restrict__ own,
                                                       const uint32_t* __restrict__ lo,
                                                       const uint32_t* __restrict__ beg,
                                                       uint32_t* __restrict__ table, uint32_t* __restrict__ place,
                                                       uint32_t* __restrict__ who) {
  __shared__ uint32_t off[kMaxColours + 1];
  const uint32_t ncol = ctr->ncolours;
  for (uint32_t c = threadIdx.x; c <= ncol; c += kBlock) off[c] = coloff[c];
  __syncthreads();
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= C) return;
  const uint32_t c = colour_of(off, ncol, k);
  const unsigned long long below = (1ull << c) - 1ull;
  const uint32_t a = ca[k], b = cb[k];
  table[start[a] + (uint32_t)__popcll(mask[a] & below)] = k;
  if (b != kNoBody) table[start[b] + (uint32_t)__popcll(mask[b] & below)] = 0x80000000u | k;
  const size_t q = (size_t)own[k] * (kMaxColours + 1) + c;
  const uint32_t j = beg[q] + (k - lo[q]);
  place[k] = j;
  who[j] = k;
}

// Where each body lives: entry of its workgroup's LDS << 2 | 1, while there are entries (most);
// else whether all its contacts are on one XCD << 1.
__global__ void __launch_bounds__(kBlock) k_flow_homes(uint32_t n, const unsigned long long* __restrict__ mask,
                                                       const uint32_t* __restrict__ start,
                                                       const uint32_t* __restrict__ table,
                                                       const uint32_t* __restrict__ own, uint32_t per_xcd,
                                                       uint32_t most, uint32_t* __restrict__ homes,
                                                       uint32_t* __restrict__ where) {
  const uint32_t b = blockIdx.x * kBlock + threadIdx.x, lane = threadIdx.x & 63;
  const uint32_t deg = b < n ? (uint32_t)__popcll(mask[b]) : 0u;
  const uint32_t* t = table + (deg ? start[b] : 0u);
  const uint32_t w = deg ? own[t[0] & 0x7FFFFFFFu] : kNoBody;
  bool one = deg > 0, near = true;
  for (uint32_t q = 1; q < deg; ++q) {
    const uint32_t v = own[t[q] & 0x7FFFFFFFu];
    one = one && v == w;
    near = near && v / per_xcd == w / per_xcd;
  }
  // Neighbouring bodies belong to few workgroups: one atomic per wave and workgroup (one per
  // body, up to a thousand on the same word, took 0.3 ms for 262,144 bodies).
  uint32_t e = most;
  for (unsigned long long todo = __ballot(one); todo;) {
    const int leader = __ffsll((long long)todo) - 1;
    const uint32_t lw = (uint32_t)__shfl((int)w, leader, 64);
    const unsigned long long same = __ballot(one && w == lw);
    uint32_t base = 0;
    if ((int)lane == leader) base = atomicAdd(&homes[lw], (uint32_t)__popcll(same));
    base = (uint32_t)__shfl((int)base, leader, 64);
    if (one && w == lw) e = base + (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
    todo &= ~same;
  }
  if (deg) where[b] = e < most ? e << 2 | 1u : near ? 2u : 0u;
}

__global__ void __launch_bounds__(kBlock) k_flow_links(uint32_t C, const uint32_t* __restrict__ ca,
                                                       const uint32_t* __restrict__ cb,
                                                       const uint32_t* __restrict__ coloff,
                                                       const StepCounters* __restrict__ ctr,
                                                       const unsigned long long* __restrict__ mask,
                                                       const uint32_t* __restrict__ start,
                                                       const uint32_t* __restrict__ table,
                                                       const uint32_t* __restrict__ place,
                                                       const uint32_t* __restrict__ where, uint2* __restrict__ from,
                                                       uint2* __restrict__ fin) {
  __shared__ uint32_t off[kMaxColours + 1];
  const uint32_t ncol = ctr->ncolours;
  for (uint32_t c = threadIdx.x; c <= ncol; c += kBlock) off[c] = coloff[c];
  __syncthreads();
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= C) return;
  const uint32_t N = flow_places(C);
  const unsigned long long below = (1ull << colour_of(off, ncol, k)) - 1ull;
  uint32_t fr[2] = {kNoBody, kNoBody}, fi[2] = {kNoBody, kNoBody};
#pragma unroll
  for (int side = 0; side < 2; ++side) {
    const uint32_t b = side ? cb[k] : ca[k];
    if (b == kNoBody) continue;
    const unsigned long long m = mask[b];
    const uint32_t wrap = (m & below) ? 0u : kFlowWrap, h = where[b];
    // colours of the contact before this one, cyclic, and of the last
    const uint32_t last = 63u - (uint32_t)__clzll((long long)m);
    const uint32_t pred = wrap ? last : 63u - (uint32_t)__clzll((long long)(m & below));
    if (h & 1u) {
      const uint32_t e = h >> 2 << (3 + kFlowColourBits) | kFlowHome;
      fr[side] = e | pred << 3 | wrap;
      fi[side] = e | last << 3;
      continue;
    }
    const uint32_t* t = table + start[b];
    const uint32_t deg = (uint32_t)__popcll(m), rank = (uint32_t)__popcll(m & below);
    auto slot = [&](uint32_t e) {
      return place[e & 0x7FFFFFFFu] + ((e >> 31) ? N : 0u) + ((h & 2u) ? 2u * N : 0u);
    };
    fr[side] = slot(t[rank ? rank - 1 : deg - 1]) << 3 | ((h & 2u) ? kFlowNear : 0u) | wrap;
    fi[side] = slot(t[deg - 1]) << 3;
  }
  from[place[k]] = make_uint2(fr[0], fr[1]);
  fin[place[k]] = make_uint2(fi[0], fi[1]);
}

// Packed records and impulses (see kRecGroups), and the scenes of an ensemble's contacts, at
// the contacts' places.
template <int D, typename Real>
__global__ void __launch_bounds__(kBlock) k_flow_pack(ContactSoA<Real> c, uint32_t C, const Real* __restrict__ body,
                                                      const uint32_t* __restrict__ place,
                                                      const uint32_t* __restrict__ cscene, Real* __restrict__ rec_,
                                                      Real* __restrict__ r_, uint32_t* __restrict__ scene) {
  using V = typename Vec4<Real>::type;
  using V2 = typename Vec2<Real>::type;
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= C) return;
  const uint32_t j = place[k];
  Rec<D, Real> R;
  load_rec<D, Real>(c, k, R);
  pack_rec<D, Real>(R, reinterpret_cast<const V*>(body), flow_places(C), j, reinterpret_cast<V*>(rec_));
  const Real* rp = c.r + 3 * (size_t)k;
  if constexpr (D == 3) reinterpret_cast<V*>(r_)[j] = V{rp[0], rp[1], rp[2], (Real)0};
  else reinterpret_cast<V2*>(r_)[j] = V2{rp[0], rp[1]};
  if (cscene) scene[j] = cscene[k];
}

hipError_t launch_flow_links(scx_ctx* c, uint32_t C, const uint32_t* ca, const uint32_t* cb, const uint32_t* first,
                             const FlowLinks& L, uint32_t xcds, uint32_t per_xcd, uint32_t home) {
  hipStream_t s = c->stream;
  const uint32_t nc = (C + kBlock - 1) / kBlock, nb = (c->n + kBlock - 1) / kBlock, G = xcds * per_xcd;
  hipError_t e = hipMemsetAsync(L.mask, 0, sizeof(unsigned long long) * ((size_t)c->n + 1), s);
  if (e != hipSuccess) return e;
  k_flow_colours<<<nc, kBlock, 0, s>>>(C, ca, cb, c->d.coloff, c->d.ctr, first, G, L.mask, L.own);
  k_flow_ranges<<<kMaxColours, kBlock, 0, s>>>(G, c->d.coloff, c->d.ctr, L.own, L.lo);
  k_flow_places<<<G, kMaxColours, 0, s>>>(per_xcd, c->d.coloff, c->d.ctr, L.lo, L.beg, L.homes);
  k_flow_offsets<<<nb, kBlock, 0, s>>>(c->n, L.mask, L.start);
  k_flow_table<<<nc, kBlock, 0, s>>>(C, ca, cb, c->d.coloff, c->d.ctr, L.mask, L.start, L.own, L.lo, L.beg, L.table,
                                      L.place, L.who);
  k_flow_homes<<<nb, kBlock, 0, s>>>(c->n, L.mask, L.start, L.table, L.own, per_xcd, home - 64, L.homes, L.where);
  k_flow_links<<<nc, kBlock, 0, s>>>(C, ca, cb, c->d.coloff, c->d.ctr, L.mask, L.start, L.table, L.place, L.where,
                                      L.from, L.fin);
  return hipGetLastError();
}

template <int D, typename Real, bool Ens, bool All>
static hipError_t launch_flow_as(scx_ctx* c, GSArgs<Real> A, FlowBufs<Real> F, uint32_t per_xcd, size_t lds,
                                 bool* launched) {
  const void* fn = (const void*)k_gs_flow<D, Real, Ens, All>;
  const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  void* args[] = {&A, &F};
  if (F.xcds * per_xcd == 1) {  // one workgroup waits for no other
    *launched = true;
    return hipLaunchKernel(fn, dim3(kXcds), dim3(kFlowThreads), args, lds, c->stream);
  }
  return launch_cooperative(c, fn, (int)(kXcds * per_xcd), kFlowThreads, args, lds, c->stream, launched);
}

template <int D, typename Real, bool Ens>
static hipError_t launch_flow_of(scx_ctx* c, GSArgs<Real> A, FlowBufs<Real> F, uint32_t per_xcd, bool* launched) {
  const uint32_t nc = (A.C + kBlock - 1) / kBlock;
  k_flow_pack<D, Real><<<nc, kBlock, 0, c->stream>>>(A.c, A.C, A.body, F.place, A.cscene, F.rec, F.r, F.scene);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  // the LDS holds the bodies that live there, and the records, links and impulses of as many
  // of a workgroup's contacts as it can
  const size_t bodies = (sizeof(Real) * FlowPort<D, Real>::NR + sizeof(uint32_t)) * F.home;
  const size_t each = sizeof(Real) * (D == 3 ? 16 + 3 : 8 + 2) + sizeof(uint2);
  // contacts of a workgroup: an equal share, and up to those of one body or one of each colour
  const uint32_t most = A.C / (F.xcds * per_xcd) + 1 + kMaxColours;
  F.rows = (most / 64 + kMaxColours + kFlowThreads / 64 + 1) / 2 * 2;
  const size_t rows = sizeof(uint2) * F.rows;
  F.kept = std::min<uint32_t>((most + 1) / 2 * 2, (uint32_t)((kFlowLdsMax - bodies - rows) / each) / 2 * 2);
  const size_t lds = bodies + rows + each * F.kept;
  return F.kept >= most ? launch_flow_as<D, Real, Ens, true>(c, A, F, per_xcd, lds, launched)
                        : launch_flow_as<D, Real, Ens, false>(c, A, F, per_xcd, lds, launched);
}

template <int D, typename Real>
hipError_t launch_gs_flow(scx_ctx* c, GSArgs<Real> A, FlowBufs<Real> F, uint32_t per_xcd, bool* launched) {
  return A.cscene ? launch_flow_of<D, Real, true>(c, A, F, per_xcd, launched)
                  : launch_flow_of<D, Real, false>(c, A, F, per_xcd, launched);
}

template hipError_t launch_gs_flow<2, float>(scx_ctx*, GSArgs<float>, FlowBufs<float>, uint32_t, bool*);
template hipError_t launch_gs_flow<3, float>(scx_ctx*, GSArgs<float>, FlowBufs<float>, uint32_t, bool*);
template hipError_t launch_gs_flow<2, double>(scx_ctx*, GSArgs<double>, FlowBufs<double>, uint32_t, bool*);
template hipError_t launch_gs_flow<3, double>(scx_ctx*, GSArgs<double>, FlowBufs<double>, uint32_t, bool*);

}  // namespace scx
