// esp_kernels.hip - HIP kernels of the per-timestep DEM engine (gfx950, FP64).
//
// Per step (launched back to back on one stream, no host synchronisation):
//   k_forces
//       the force laws of every interaction group in one launch (one block
//       segment per group), one thread per interaction; each writes its share
//       into both particles' slots.  In a queued step block 0 meanwhile applies
//       the previous step's bond breaks and appends the new pairs of the
//       flagged particles (and computes their forces)
//   k_gather_integrate (k_gather_wide for many particles, k_gather_stress where
//       particle stresses are kept)
//       per particle: wall and body forces, then the records of its
//       interactions in a fixed order (CSR), then the CParticle/CRotParticle
//       first-order update and the max-displacement reduction; wall-force
//       partials of every 64 particles
//   k_contact_step, k_contact_block
//       instead of these two where no group is bonded and one launch is faster
//       (the host step's fused_form): each particle evaluates its side of its
//       interactions and integrates
//   k_batch_end (once per queued batch)
//       fixed-order sums of the wall-force partials of every step of the batch,
//       written with the batch's status to page-locked host memory
// Every per-step kernel first evaluates the previous step's status; if that
// step displaced a particle by more than verletDist/2 or broke a bond, the host
// must do bookkeeping first, so the kernel records the halt and returns, and
// all later queued steps return too.
//
// Rebuild / update kernels (launched from the host's bookkeeping path):
//   cell binning (counting sort + per-cell ordering), candidate pair search over
//   the 27-cell neighbourhood emitting pairs sorted by (id1, id2), interaction
//   storage updates (history carried over by key lookup), bond removal,
//   wall candidate refresh and the per-particle CSR of force records.
#include <cstring>
#include <hip/hip_ext.h>

#include "esp_internal.h"
#include "esp_math.h"
#include "esp_wave.h"

#define BS 256
static inline int nblk(long long n, int bs = BS) { return (int)((n + bs - 1) / bs); }

__device__ __forceinline__ dv3 xyz(double4 a) { return mk3(a.x, a.y, a.z); }

__device__ __forceinline__ bool step_skip(const StepCtl& c)
{
  if (!c.guarded) return false;
  const int halted = *(volatile int*)c.halted;
  const unsigned long long md = c.prev->maxdisp2;  // both loads in flight together
  if (halted) return true;
  if (md > c.thresh) {  // neighbour table must be rebuilt: host bookkeeping
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      *c.reason = 1;
      *c.halted = c.step_id;
    }
    return true;
  }
  return false;
}

// The image of particle 2 nearest to particle 1 in a circular x dimension:
// shifted by the period when the two are more than half a period apart, one
// addition, as a ghost copy carries its shifted position (CParticle::setCircular,
// Particle.cpp:336-342); period 0: not circular.
__device__ __forceinline__ double4 x_image(double4 P1, double4 P2, double period)
{
  if (period > 0.0) {
    const double d = P1.x - P2.x;
    if (d > 0.5 * period) P2.x = P2.x + period;
    else if (d < -0.5 * period) P2.x = P2.x - period;
  }
  return P2;
}

__device__ __forceinline__ long long pair_key(int a, int b)
{
  return (long long)(((unsigned long long)(unsigned)a << 32) | (unsigned long long)(unsigned)b);
}

// ---------------------------------------------------------------------------
// pair-key hash sets (linear probing; bounded probes)
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned hs_slot(unsigned long long k, unsigned mask)
{
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  k *= 0xc4ceb9fe1a85ec53ull;
  k ^= k >> 33;
  return (unsigned)k & mask;
}
__device__ __forceinline__ int hs_find(HashRef h, long long key)
{
  const unsigned long long k = (unsigned long long)key;
  unsigned s = hs_slot(k, h.mask);
  for (unsigned probe = 0; probe <= h.mask; probe++) {
    const unsigned long long v = h.t[s];
    if (v == k) return (int)s;
    if (v == HS_EMPTY) return -1;
    s = (s + 1) & h.mask;
  }
  return -1;
}
__device__ __forceinline__ void hs_insert(HashRef h, long long key)
{
  const unsigned long long k = (unsigned long long)key;
  unsigned s = hs_slot(k, h.mask);
  for (unsigned probe = 0; probe <= h.mask; probe++) {
    const unsigned long long old = atomicCAS(&h.t[s], HS_EMPTY, k);
    if (old == HS_EMPTY || old == k) return;
    s = (s + 1) & h.mask;
  }
}
__device__ __forceinline__ void hs_erase(HashRef h, long long key)
{
  const int s = hs_find(h, key);
  if (s >= 0) h.t[s] = HS_TOMB;
}
__device__ __forceinline__ bool excluded(const ExclSet& ex, long long key)
{
  for (int x = 0; x < ex.count; x++)
    if (hs_find(ex.h[x], key) >= 0) return true;
  return false;
}

// a candidate pair (particle slots a, b; id key) the group does not take
__device__ __forceinline__ bool rejected(const ExclSet& ex, long long key, int a, int b)
{
  if (ex.tagged) {
    int t1 = ex.tag[a], t2 = ex.tag[b];
    if (t1 > t2) {
      const int th = t1;
      t1 = t2;
      t2 = th;
    }
    if (!(((t1 & ex.mask1) == (ex.tag1 & ex.mask1)) && ((t2 & ex.mask2) == (ex.tag2 & ex.mask2))))
      return true;
  }
  return excluded(ex, key);
}

// ---------------------------------------------------------------------------
// per-step interaction kernels
// ---------------------------------------------------------------------------
// Each interaction writes its result per side straight into the two
// particles' CSR slots: force and moment on that particle (and, with stresses
// tracked, the contact point relative to it).  Slot positions are fixed at each
// rebuild (slot_of), so a particle later reads one contiguous run.
__device__ __forceinline__ void put3(double* d, dv3 v)
{
  d[0] = v.x;
  d[1] = v.y;
  d[2] = v.z;
}
__device__ __forceinline__ void zero_slot(double* d, int ss)
{
  for (int k = 0; k < ss; k++) d[k] = 0.0;
}
// contact point p2 + r2 / (r1 + r2) (p1 - p2) of the pair laws
// (ARotBondedInteraction.cpp:437-440, RotFricInteraction.cpp:185, ElasticInteraction.cpp:61),
// stored relative to each particle
__device__ __forceinline__ void put_rel(double* a, double* b, double4 P1, double4 P2)
{
  const dv3 D = sub3(xyz(P1), xyz(P2));
  const dv3 c = add3(xyz(P2), mul3(D, P2.w / (P1.w + P2.w)));
  put3(a + 6, sub3(c, xyz(P1)));
  put3(b + 6, sub3(c, xyz(P2)));
}

// A bond's particle pair read with one 8-byte load.  The incremental update
// that runs beside the force blocks (block 0 of a queued step) marks the bonds
// broken in the previous step dead by storing (-1, -1) over their pairs.  A
// plain int2 read may be compiled into two 4-byte loads, the second issued
// only after the first index passed its test, and could then return a live
// first index with the dead second one (and the force law would gather
// position -1).  One relaxed atomic load returns either the whole old pair or
// (-1, -1).
__device__ __forceinline__ int2 load_pair_once(const int2* a)
{
  const unsigned long long v =
      __hip_atomic_load(reinterpret_cast<unsigned long long*>(const_cast<int2*>(a)),
                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  return make_int2((int)(unsigned)(v & 0xffffffffull), (int)(unsigned)(v >> 32));
}

// ARotBondedInteraction::calcForces + CRotBondedInteraction::broken
// (ARotBondedInteraction.cpp:307-448, RotBondedInteraction.cpp:175-219)
__device__ __forceinline__ void rot_bond_item(const StepCtl& ctl, const PView& p, int b,
                                              const ForceSeg& g, const ForceLaunch& fl)
{
  const int nb = g.n;
  const int2* __restrict__ ij = g.ij;
  if (b >= nb) return;
  const int2 e = load_pair_once(ij + b);
  const int2 so = fl.slot_of[g.rec_off + b];
  if (e.x < 0 || e.y < 0) return;  // broken earlier: removed from the group, slots left at zero
  const double4 P1 = p.pos[e.x], P2 = x_image(P1, p.pos[e.y], fl.period);
  const double4 Q1 = p.quat[e.x], Q2 = p.quat[e.y];
  const double4 K = g.k4[b], D = g.D4[b];
  // broken in an earlier step (D.w holds that step): the incremental update
  // that runs beside this launch removes the bond and clears its slots
  if (D.w != 0.0 && D.w < fl.step) return;
  BondResult o;
  esp_rot_bond_law(xyz(P1), dquat{Q1.x, mk3(Q1.y, Q1.z, Q1.w)}, P1.w, xyz(P2),
                   dquat{Q2.x, mk3(Q2.y, Q2.z, Q2.w)}, P2.w, K.x, K.y, K.z, K.w, xyz(D), o);
  // the strengths are needed only by the break test after the law: loaded
  // here, their latency overlaps the slot stores
  const double4 M = g.mx4[b];
  double* s0 = fl.slots + (size_t)fl.ss * so.x;
  double* s1 = fl.slots + (size_t)fl.ss * so.y;
  put3(s0, o.f1);
  put3(s0 + 3, o.m1);
  put3(s1, neg3(o.f1));
  put3(s1 + 3, o.m2);
  if (fl.ss == 9) put_rel(s0, s1, P1, P2);
  fl.sact[so.x] = 1;
  fl.sact[so.y] = 1;
  // CRotBondedInteraction::getCriterion (RotBondedInteraction.cpp:221-227)
  if (fl.crit)
    fl.crit[g.bond_off + b] = o.nForce / M.x + o.shForce / M.y + o.tMoment / M.z + o.bMoment / M.w;
  if (g.sc) return;  // broken by the particle stresses after the integration
  if (esp_bond_broken(o.nForce, o.shForce, o.tMoment, o.bMoment, M.x, M.y, M.z, M.w, g.truncated,
                      g.beta1, g.beta2)) {
    g.D4[b].w = fl.step;
    const int slot = atomicAdd(&ctl.cur->nbroken, 1);
    fl.broken_list[slot] = g.bond_off + b;
  }
}

__device__ __forceinline__ int record_of(int c, int nc, int rec_off, int app_rec_off)
{
  return c < nc ? rec_off + c : app_rec_off + (c - nc);
}

// CRotFrictionInteraction::calcForces (RotFricInteraction.cpp:103-231)
// RIGID: the launch may hold rigid=True groups (their law is only compiled into
// the kernel that handles them, so the common kernel keeps its registers)
template <bool RIGID>
__device__ __forceinline__ void rot_friction_item(const PView& p, int c, const ForceSeg& g,
                                                  const ForceLaunch& fl)
{
  const int nc = g.n;
  const int2 e = g.ij[c];
  const int rec = record_of(c, nc, g.rec_off, g.app_rec_off);
  const double4 P1 = p.pos[e.x], P2 = x_image(P1, p.pos[e.y], fl.period);
  const double4 st = g.ff[c];
  const dv3 Dq = sub3(xyz(P1), xyz(P2));
  const double eq = P1.w + P2.w;
  if (!(dot3(Dq, Dq) < (eq * eq))) {
    // not touching: history cleared, no force.  A pair that did not touch in
    // the last step already holds zero slots; once both history buffers hold
    // zero (flag bit 2) nothing is written (nor are its slots looked up).
    const int fw = (int)st.w;
    if ((fw & 3) != 0 || st.x != 0.0 || st.y != 0.0 || st.z != 0.0) {
      const int2 so = fl.slot_of[rec];
      g.ff_out[c] = make_double4(0.0, 0.0, 0.0, 0.0);
      zero_slot(fl.slots + (size_t)fl.ss * so.x, fl.ss);
      zero_slot(fl.slots + (size_t)fl.ss * so.y, fl.ss);
      fl.sact[so.x] = 0;
      fl.sact[so.y] = 0;
    } else if (!(fw & 4)) {
      g.ff[c] = make_double4(0.0, 0.0, 0.0, 4.0);
      g.ff_out[c] = make_double4(0.0, 0.0, 0.0, 4.0);
    }
    return;
  }
  // touching: the slot lookup goes out with the velocity loads
  const int2 so = fl.slot_of[rec];
  double* s0 = fl.slots + (size_t)fl.ss * so.x;
  double* s1 = fl.slots + (size_t)fl.ss * so.y;
  const double4 V1 = p.vel[e.x], V2 = p.vel[e.y], W1 = p.ang[e.x], W2 = p.ang[e.y];
  double kk, kks;
  esp_friction_k(g.k, g.ks, g.scaling, g.meanR, P1.w, P2.w, fl.do2d, kk, kks);
  dv3 ffr = mk3(st.x, st.y, st.z);
  bool slipping = (((int)st.w) & 1) != 0;
  dv3 f1, m1, m2;
  if (RIGID && g.rigid)
    esp_rot_friction_rigid_law(xyz(P1), xyz(V1), xyz(W1), P1.w, xyz(P2), xyz(V2), xyz(W2), P2.w,
                               kk, kks, g.mu_d, g.mu_s, fl.dt, (((int)st.w) & 2) != 0, ffr,
                               slipping, f1, m1, m2);
  else
    esp_rot_friction_law(xyz(P1), xyz(V1), xyz(W1), P1.w, xyz(P2), xyz(V2), xyz(W2), P2.w, kk,
                         kks, g.mu_d, g.mu_s, fl.dt, ffr, slipping, f1, m1, m2);
  g.ff_out[c] = make_double4(ffr.x, ffr.y, ffr.z, (double)((slipping ? 1 : 0) | 2));
  put3(s0, f1);
  put3(s0 + 3, m1);
  put3(s1, neg3(f1));
  put3(s1 + 3, m2);
  if (fl.ss == 9) put_rel(s0, s1, P1, P2);
  fl.sact[so.x] = 1;
  fl.sact[so.y] = 1;
}

// CElasticInteraction::calcForces (ElasticInteraction.cpp:54-71); no moments
// (their slot parts stay zero)
__device__ __forceinline__ void nrot_elastic_item(const PView& p, int c, const ForceSeg& g,
                                                  const ForceLaunch& fl)
{
  const int nc = g.n;
  const int2 e = g.ij[c];
  const int2 so = fl.slot_of[record_of(c, nc, g.rec_off, g.app_rec_off)];
  const double4 P1 = p.pos[e.x], P2 = x_image(P1, p.pos[e.y], fl.period);
  double* s0 = fl.slots + (size_t)fl.ss * so.x;
  double* s1 = fl.slots + (size_t)fl.ss * so.y;
  const dv3 D = sub3(xyz(P1), xyz(P2));
  double dist = dot3(D, D);
  const double eq_dist = P1.w + P2.w;
  if (dist < (eq_dist * eq_dist)) {
    const double kk = esp_elastic_k(g.k, g.scaling, P1.w, P2.w, fl.do2d);
    dist = sqrt(dist);
    const dv3 force = mul3(D, kk * (dist - eq_dist) / dist);
    put3(s0, neg3(force));
    put3(s1, force);
    if (fl.ss == 9) put_rel(s0, s1, P1, P2);
    fl.sact[so.x] = 1;
    fl.sact[so.y] = 1;
  } else {
    put3(s0, mk3(0.0, 0.0, 0.0));
    put3(s1, mk3(0.0, 0.0, 0.0));
    fl.sact[so.x] = 0;
    fl.sact[so.y] = 0;
  }
}

// CRotElasticInteraction::calcForces (RotElasticInteraction.cpp:69-88)
__device__ __forceinline__ void rot_elastic_item(const PView& p, int c, const ForceSeg& g,
                                                 const ForceLaunch& fl)
{
  const int nc = g.n;
  const int2 e = g.ij[c];
  const int2 so = fl.slot_of[record_of(c, nc, g.rec_off, g.app_rec_off)];
  const double4 P1 = p.pos[e.x], P2 = x_image(P1, p.pos[e.y], fl.period);
  double* s0 = fl.slots + (size_t)fl.ss * so.x;
  double* s1 = fl.slots + (size_t)fl.ss * so.y;
  const dv3 rb = sub3(xyz(P1), xyz(P2));
  const double rbNorm = norm3(rb);
  const double r_0Norm = P1.w + P2.w;
  if (rbNorm < r_0Norm) {
    const dv3 delta_r = div3(mul3(rb, rbNorm - r_0Norm), rbNorm);
    const dv3 force = mul3(delta_r, esp_rotelastic_k(g.k, g.scaling, P1.w, P2.w, fl.do2d));
    put3(s0, neg3(force));
    put3(s1, force);
    if (fl.ss == 9) put_rel(s0, s1, P1, P2);
    fl.sact[so.x] = 1;
    fl.sact[so.y] = 1;
  } else {
    put3(s0, mk3(0.0, 0.0, 0.0));
    put3(s1, mk3(0.0, 0.0, 0.0));
    fl.sact[so.x] = 0;
    fl.sact[so.y] = 0;
  }
}

// NeighborTable::index (ntable.hpp:128-139): floor((x - x0)/dim) - global index,
// with values outside the int range (and NaN) mapped to "outside" as x86's
// conversion does.
__device__ __forceinline__ bool cell_coords(const GridParams& g, double x, double y, double z,
                                            int& ix, int& iy, int& iz)
{
  const double fx = floor((x - g.x0) / g.dim);
  const double fy = floor((y - g.y0) / g.dim);
  const double fz = floor((z - g.z0) / g.dim);
  if (!(fx >= -2147483648.0 && fx < 2147483648.0 && fy >= -2147483648.0 && fy < 2147483648.0 &&
        fz >= -2147483648.0 && fz < 2147483648.0))
    return false;
  ix = (int)fx - g.gx;
  iy = (int)fy - g.gy;
  iz = (int)fz - g.gz;
  // circular x: positions are wrapped into [x0, x0 + L) at each rebuild; a
  // rounding of (x - x0)/dim onto the end of the range stays in the last cell
  if (g.circ_x && x >= g.x0 && x < g.x0 + g.period) ix = ix < 0 ? 0 : (ix >= g.nx ? g.nx - 1 : ix);
  return true;
}

// CBondedWallInteraction::calcForces (BWallInteraction.hpp:35-52): the force on
// the particle, -(total displacement of the particle - that of the wall) k',
// k' = k pi r (3-D; the constant of BWallInteraction.hpp:25-31) or k (2-D)
__device__ __forceinline__ dv3 bonded_wall_force(const WallParam& W, dv3 x, dv3 x_init, double r,
                                                 int do2d)
{
  const double scale = do2d ? 1.0 : 3.1415926536 * r;
  const double kb = W.k * scale;
  const dv3 D = sub3(sub3(x, x_init), mk3(W.disp[0], W.disp[1], W.disp[2]));
  return mul3(mul3(D, kb), -1.0);
}

// Wall-group membership and inner flags of one particle (CEWallInteractionGroup::
// Update, EWallInteractionGroup.hpp:57-82, with isInInner, ntable.hpp:207-222).
__device__ __forceinline__ unsigned wall_membership(const GridParams& g, int nwg,
                                                    const WallParam* W, double4 P, unsigned fl)
{
  fl &= ~((0xFFu << PF_WALL_SHIFT) | (0xFFu << PF_INNER_SHIFT));
  int ix = 0, iy = 0, iz = 0;
  bool inner = false;
  if (cell_coords(g, P.x, P.y, P.z, ix, iy, iz)) {
    // circular x: no padding cells in x, every x is inner
    const bool xin = g.circ_x || ((ix > 0) && (ix < g.nx - 1));
    if (g.nz < 3) inner = xin && (iy > 0) && (iy < g.ny - 1);
    else inner = xin && (iy > 0) && (iy < g.ny - 1) && (iz > 0) && (iz < g.nz - 1);
  }
  for (int w = 0; w < nwg; w++) {
    const dv3 n = mk3(W[w].nrm[0], W[w].nrm[1], W[w].nrm[2]);
    const double dist = dot3(sub3(xyz(P), mk3(W[w].o[0], W[w].o[1], W[w].o[2])), n);
    if (fabs(dist) < g.dim) {
      fl |= 1u << (PF_WALL_SHIFT + w);
      if (inner) fl |= 1u << (PF_INNER_SHIFT + w);
    }
  }
  return fl;
}

// ---------------------------------------------------------------------------
// gather + integrate
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v)
{
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long w = __shfl_xor(v, o, 64);
    v = w > v ? w : v;
  }
  return v;
}

// Fixed-order sum of (a, b, c) over the block, valid in thread 0: within each
// wave, then the waves in index order.  Every thread of the block must call it.
__device__ __forceinline__ void block_sum3(double& a, double& b, double& c, double* lds)
{
  a = wave_sum(a);
  b = wave_sum(b);
  c = wave_sum(c);
  __syncthreads();  // lds free from the previous call
  if ((threadIdx.x & 63) == 0) {
    const int w = threadIdx.x >> 6;
    lds[3 * w] = a;
    lds[3 * w + 1] = b;
    lds[3 * w + 2] = c;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w = 1; w < BS / 64; w++) {
      a = a + lds[3 * w];
      b = b + lds[3 * w + 1];
      c = c + lds[3 * w + 2];
    }
}

// sigma(i,j) -= f_i rel_j (CParticle::applyForce, Particle.cpp:391-400)
__device__ __forceinline__ void stress_add(double (&sg)[3][3], dv3 f, dv3 rel)
{
  const double fv[3] = {f.x, f.y, f.z}, rv[3] = {rel.x, rel.y, rel.z};
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++) sg[i][j] -= fv[i] * rv[j];
}

// Wall interaction groups, name order (EWallInteraction.hpp:42-78), then body
// forces, name order (BodyForceGroup.hpp:41-65): the force the particle's
// interactions are added to.  In a bonded group the tagged candidates are
// bonded instead.  flw: the particle's flags; i: its slot.
// STRESS: every applied force also updates the particle's stress sum, in the
// order the forces are summed.  EXTRA: damping groups, bonded or tagged walls
// exist (kept out of the plain kernels).
template <bool STRESS, bool EXTRA>
__device__ __forceinline__ dv3 wall_body_force(const GatherParams& gp, int i, unsigned flw, dv3 x,
                                               double r, double mass, double (&sg)[3][3])
{
  dv3 F = mk3(0.0, 0.0, 0.0);
  const bool any = __ballot(((flw >> PF_WALL_SHIFT) & 0xFFu) != 0u) != 0ull;  // of the wave
  for (int w = 0; any && w < gp.nwg; w++) {
    if (!((flw >> (PF_WALL_SHIFT + w)) & 1u)) continue;
    const WallParam& W = gp.wall[w];
    if (EXTRA && W.tagged && !((flw >> (PF_BTAG_SHIFT + w)) & 1u)) continue;
    if (EXTRA && W.bonded && ((flw >> (PF_BTAG_SHIFT + w)) & 1u)) {
      const dv3 fb = bonded_wall_force(W, x, xyz(gp.init[i]), r, gp.do2d);
      F = add3(F, fb);
      if (STRESS) stress_add(sg, fb, sub3(x, x));
      continue;
    }
    const dv3 n = mk3(W.nrm[0], W.nrm[1], W.nrm[2]);
    const double dist = dot3(sub3(x, mk3(W.o[0], W.o[1], W.o[2])), n);
    if (dist < r) {
      double f = 1.0;
      if (!gp.do2d) f *= 3.141592654 * r;
      const dv3 force = mul3(n, (f * W.k) * (r - dist));
      F = add3(F, force);
      if (STRESS) stress_add(sg, force, sub3(sub3(x, mul3(n, dist)), x));
    }
  }
  // applied at the centre
  for (int g = 0; g < gp.ngrav; g++) {
    const dv3 fg = mul3(mk3(gp.g[g][0], gp.g[g][1], gp.g[g][2]), mass);
    F = add3(F, fg);
    if (STRESS) stress_add(sg, fg, sub3(x, x));
  }
  return F;
}

// The wall force on an inner candidate of wall group w, as wall_body_force
// applies it (the wall forces sum these; zero for every other particle)
template <bool EXTRA>
__device__ __forceinline__ dv3 wall_share(const GatherParams& gp, int w, int i, unsigned flw, dv3 x,
                                          double r)
{
  if (!((flw >> (PF_WALL_SHIFT + w)) & 1u) || !((flw >> (PF_INNER_SHIFT + w)) & 1u))
    return mk3(0.0, 0.0, 0.0);
  const WallParam& W = gp.wall[w];
  // untagged candidates of a tagged elastic wall: no interaction
  if (EXTRA && W.tagged && !((flw >> (PF_BTAG_SHIFT + w)) & 1u)) return mk3(0.0, 0.0, 0.0);
  // CWall::addForce(force) subtracts the bonded force: the particle's share
  if (EXTRA && W.bonded && ((flw >> (PF_BTAG_SHIFT + w)) & 1u))
    return bonded_wall_force(W, x, xyz(gp.init[i]), r, gp.do2d);
  const dv3 n = mk3(W.nrm[0], W.nrm[1], W.nrm[2]);
  const double dist = dot3(sub3(x, mk3(W.o[0], W.o[1], W.o[2])), n);
  if (!(dist < r)) return mk3(0.0, 0.0, 0.0);
  double f = 1.0;
  if (!gp.do2d) f *= 3.141592654 * r;
  return mul3(n, (f * W.k) * (r - dist));
}

// Damping groups, last (SubLattice.hpp:2143-2147), in their map order, then the
// CParticle / CRotParticle update of particle i; writes its new state to po
// (the arrays it is stepped into) and returns |x - x_old|^2.
template <bool STRESS, bool EXTRA>
__device__ __forceinline__ double damp_and_integrate(const PView& po, const GatherParams& gp, int i,
                                                     unsigned fl, dv3 F, dv3 M, double4 P, double4 Vv,
                                                     double4 O, double4 A, double4 Q,
                                                     double (&sg)[3][3])
{
  dv3 x = xyz(P), v = xyz(Vv);
  const double r = P.w, invm = Vv.w, mass = O.w;
  const double dt = gp.dt;
  for (int d = 0; EXTRA && d < gp.ndamp; d++) {
    const int ty = gp.damp_type[d];
    const double visc = gp.damp_visc[d];
    if (ty == ESP_DAMPING || ty == ESP_ROT_DAMPING) {
      const bool rd = ty == ESP_ROT_DAMPING;
      const double mi = rd ? gp.inert[i] : mass;
      const dv3 vr = esp_damping_vrel(rd ? xyz(A) : v, rd ? M : F, rd ? A.w : invm, mi, visc, dt,
                                      gp.damp_maxit[d]);
      const dv3 fd = mul3(mul3(vr, -1.0 * visc), mi);
      if (rd) {
        M = add3(M, fd);
      } else {
        F = add3(F, fd);
        if (STRESS) stress_add(sg, fd, sub3(x, x));
      }
    } else {
      const bool rd = ty == ESP_ROT_LOCAL_DAMPING;
      const dv3 vv = rd ? xyz(A) : v, ff = rd ? M : F;
      const dv3 fd = mul3(mk3(esp_local_damping_c(ff.x, vv.x), esp_local_damping_c(ff.y, vv.y),
                              esp_local_damping_c(ff.z, vv.z)),
                          -1.0 * visc);
      if (rd) {
        M = add3(M, fd);
      } else {
        F = add3(F, fd);
        if (STRESS) stress_add(sg, fd, sub3(x, x));
      }
    }
  }
  if (gp.rot) {
    dv3 w = xyz(A);
    dquat q = dquat{Q.x, mk3(Q.y, Q.z, Q.w)};
    if (fl & PF_ROT) {
      if (gp.do2d) {
        F = mk3(F.x, F.y, 0);
        M = mk3(0, 0, M.z);
      }
      w = add3(w, mul3(M, dt * A.w));
      const dquat dq = qmul4(dquat{0, w}, q);
      const double h = dt / 2.0;
      q.s += h * dq.s;
      q.v = add3(q.v, mul3(dq.v, h));
    } else {
      w = mk3(0.0, 0.0, 0.0);
    }
    if (fl & PF_DYN) {
      if (gp.do2d) F = mk3(F.x, F.y, 0);
      v = add3(v, mul3(mul3(F, invm), dt));
      x = add3(x, mul3(v, dt));
    }
    const double module = sqrt(q.s * q.s + q.v.x * q.v.x + q.v.y * q.v.y + q.v.z * q.v.z);
    if (module != 0.0) {
      const double inverse = 1.0 / module;
      q.s = inverse * q.s;
      q.v = mul3(q.v, inverse);
    }
    po.ang[i] = make_double4(w.x, w.y, w.z, A.w);
    po.quat[i] = make_double4(q.s, q.v.x, q.v.y, q.v.z);
    if (gp.store_fm) po.mom[i] = make_double4(M.x, M.y, M.z, 0.0);
  } else if (fl & PF_DYN) {
    if (gp.do2d) F = mk3(F.x, F.y, 0);
    v = add3(v, mul3(mul3(F, invm), dt));
    x = add3(x, mul3(v, dt));
  }
  po.pos[i] = make_double4(x.x, x.y, x.z, r);
  po.vel[i] = make_double4(v.x, v.y, v.z, invm);
  if (gp.store_fm) po.frc[i] = make_double4(F.x, F.y, F.z, 0.0);
  if (STRESS) {
    double* o = gp.sig + 9 * (size_t)i;
    for (int a = 0; a < 3; a++)
      for (int b = 0; b < 3; b++) o[3 * a + b] = sg[a][b];
  }
  const dv3 d = sub3(x, xyz(O));
  return dot3(d, d);
}

// The gather of an engine that accumulates particle stresses: slots carry contact
// points (9 doubles)
template <bool EXTRA>
__global__ __launch_bounds__(BS) void k_gather_stress(StepCtl ctl, PView p, GatherParams gp)
{
  constexpr int GATHER_CHUNK = 2;
  double sg[3][3];
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 3; j++) sg[i][j] = 0.0;
  if (step_skip(ctl)) return;
  __shared__ double lds3[3 * (BS / 64)];
  __shared__ unsigned long long mred[BS / 64];
  // pairs appended by this step's incremental update are covered by the force
  // blocks from the next step on
  if (gp.n_app && blockIdx.x == 0 && threadIdx.x == 0) gp.n_app[1] = gp.n_app[0];
  const int i = blockIdx.x * BS + threadIdx.x;
  const bool act = i < p.n;
  const int ii = act ? i : 0;
  // every load that does not depend on another is issued here, together
  const double4 P = p.pos[ii];
  const unsigned fl = p.flags[ii];
  const double4 Vv = p.vel[ii];
  const double4 O = p.old[ii];
  const int e0 = gp.inc_off[ii], e1 = gp.inc_off[ii + 1];
  const int xcnt = gp.xcnt[ii];
  double4 A = make_double4(0.0, 0.0, 0.0, 0.0), Q = A;
  if (gp.rot) {
    A = p.ang[ii];
    Q = p.quat[ii];
  }
  const int refresh = gp.nwg > 0 && ctl.guarded && ctl.prev->nbroken > 0;
  const dv3 x0 = xyz(P);
  const double r = P.w;
  unsigned flw = fl;
  if (act && refresh) {
    // bonds broke in the previous step: the reference's updateInteractions
    // re-Updates the wall groups (EWallInteractionGroup.hpp:57-82) before forces
    flw = wall_membership(gp.grid, gp.nwg, gp.wall, P, fl);
    p.flags[i] = flw;
  }
  unsigned long long md = 0;
  if (act) {
    dv3 F = wall_body_force<true, EXTRA>(gp, i, flw, x0, r, O.w, sg);
    dv3 M = mk3(0.0, 0.0, 0.0);
    // the particle's slots in summation order (its CSR run, then its appendix
    // slots), fetched GATHER_CHUNK at a time so their loads are in flight
    // together; the sum itself stays sequential.  Moments of laws without
    // moments are zeros, and a sum that starts at +0 never becomes -0, so
    // adding them changes nothing.
    const int nmain = e1 - e0;
    const int cnt = nmain + xcnt;
    for (int b = 0; b < cnt; b += GATHER_CHUNK) {
      dv3 f[GATHER_CHUNK], m[GATHER_CHUNK], rl[GATHER_CHUNK];
#pragma unroll
      for (int k = 0; k < GATHER_CHUNK; k++) {
        const int t = b + k;
        const int slot = t >= cnt ? 0 : t < nmain ? e0 + t : gp.xbase + ESP_XSLOTS * i + (t - nmain);
        const double* q = gp.slots + (size_t)9 * slot;
        f[k] = mk3(q[0], q[1], q[2]);
        m[k] = mk3(q[3], q[4], q[5]);
        rl[k] = mk3(q[6], q[7], q[8]);
      }
#pragma unroll
      for (int k = 0; k < GATHER_CHUNK; k++) {
        if (b + k >= cnt) break;
        F = add3(F, f[k]);
        stress_add(sg, f[k], rl[k]);
        M = add3(M, m[k]);
      }
    }
    md = (unsigned long long)__double_as_longlong(
        damp_and_integrate<true, EXTRA>(p, gp, i, fl, F, M, P, Vv, O, A, Q, sg));
  }
  // max displacement: wave, then block, then one atomic per block
  md = wave_max_u64(md);
  if ((threadIdx.x & 63) == 0) mred[threadIdx.x >> 6] = md;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long m = mred[0];
    for (int w = 1; w < BS / 64; w++) m = mred[w] > m ? mred[w] : m;
    // only "beyond verletDist/2" is ever read, so smaller maxima need no atomic
    if (m > ctl.thresh) atomicMax(&ctl.cur->maxdisp2, m);
  }
  // this block's partial of each wall force: the forces on inner particles,
  // recomputed from the same values as above, in a fixed-order block sum;
  // a block without wall candidates writes zeros
  const unsigned wall_bits = act ? (flw >> PF_WALL_SHIFT) & 0xFFu : 0u;
  const int any_wall = gp.nwg > 0 ? __syncthreads_or(wall_bits != 0u) : 0;
  for (int w = 0; w < gp.nwg; w++) {
    if (!any_wall) {
      if (threadIdx.x == 0) {
        double* q = gp.wall_part + ((size_t)blockIdx.x * gp.nwg + w) * 3;
        q[0] = 0.0; q[1] = 0.0; q[2] = 0.0;
      }
      continue;
    }
    const dv3 sh = act ? wall_share<EXTRA>(gp, w, i, flw, x0, r) : mk3(0.0, 0.0, 0.0);
    double wx = sh.x, wy = sh.y, wz = sh.z;
    block_sum3(wx, wy, wz, lds3);
    if (threadIdx.x == 0) {
      double* q = gp.wall_part + ((size_t)blockIdx.x * gp.nwg + w) * 3;
      q[0] = wx; q[1] = wy; q[2] = wz;
    }
  }
}

// The end of a batch of steps, the one launch the host waits for.  Block s sums
// step s's wall partials in a fixed order (LIST: the 64-particle groups named in
// list, else every block's) straight into page-locked host memory, so no copy
// follows; slots of steps that were skipped hold stale values the host does not
// read.  Block 0 also reports why the queue halted and the last completed
// step's status, and clears every other entry of the ring and the halt mark for
// the next batch.  With three copies into pageable memory and two launches around a
// batch a batch of one step of 97 particles took 72 us; with this 38.
template <bool LIST>
__global__ __launch_bounds__(BS) void k_batch_end(BatchEnd be)
{
  __shared__ double lds3[3 * (BS / 64)];
  const int nb = LIST ? *be.list_n : be.nblocks;
  const double* ps = be.part + (size_t)blockIdx.x * be.nblocks * be.nwg * 3;
  for (int w = 0; w < be.nwg; w++) {
    double a = 0.0, b = 0.0, c = 0.0;
    for (int k = threadIdx.x; k < nb; k += BS) {
      const double* q = ps + ((size_t)(LIST ? be.list[k] : k) * be.nwg + w) * 3;
      a = a + q[0];
      b = b + q[1];
      c = c + q[2];
    }
    block_sum3(a, b, c, lds3);
    if (threadIdx.x == 0) {
      double* o = be.walls + ((size_t)blockIdx.x * be.nwg + w) * 3;
      o[0] = a;
      o[1] = b;
      o[2] = c;
    }
  }
  if (blockIdx.x != 0) return;
  const int halted = *be.halted;
  __syncthreads();  // every thread has the mark before it is cleared
  const int done = halted ? halted - 1 : be.nsteps;
  const int last = (int)((be.step0 + done - 1) % be.ring_size);
  for (int t = threadIdx.x; t < be.ring_size; t += BS) {
    StepStatus& st = be.ring[t];
    if (t == last) {
      be.out->maxdisp2 = st.maxdisp2;
      be.out->nbroken = st.nbroken;
    } else {
      st.maxdisp2 = 0ull;
      st.nbroken = 0;
      st.pad = 0;
    }
  }
  if (threadIdx.x == 0) {
    be.out->halted = halted;
    be.out->reason = *be.reason;
    *be.halted = 0;
  }
}

// ---------------------------------------------------------------------------
// one whole step of an engine without bonded groups
// ---------------------------------------------------------------------------
// bits of the four lanes of a group of 4
__device__ __forceinline__ unsigned long long group_or(unsigned long long v)
{
  int lo = (int)(v & 0xffffffffull), hi = (int)(v >> 32);
  lo |= __builtin_amdgcn_mov_dpp(lo, 0xB1, 0xf, 0xf, true);  // lanes 1,0,3,2
  hi |= __builtin_amdgcn_mov_dpp(hi, 0xB1, 0xf, 0xf, true);
  lo |= __builtin_amdgcn_mov_dpp(lo, 0x4E, 0xf, 0xf, true);  // lanes 2,3,0,1
  hi |= __builtin_amdgcn_mov_dpp(hi, 0x4E, 0xf, 0xf, true);
  return ((unsigned long long)(unsigned)hi << 32) | (unsigned long long)(unsigned)lo;
}

// A RotFriction pair apart, as its first particle sees it: history cleared; once
// both buffers hold zero (flag bit 2) nothing is written.
__device__ __forceinline__ void clear_history(const ContactSeg& g, int c)
{
  const double4 st = g.ff[c];
  const int fw = (int)st.w;
  if ((fw & 3) != 0 || st.x != 0.0 || st.y != 0.0 || st.z != 0.0) {
    g.ff_out[c] = make_double4(0.0, 0.0, 0.0, 0.0);
  } else if (!(fw & 4)) {
    g.ff[c] = make_double4(0.0, 0.0, 0.0, 4.0);
    g.ff_out[c] = make_double4(0.0, 0.0, 0.0, 4.0);
  }
}

// the group of a record (KIND: the launch's only group, or 0)
template <int KIND>
__device__ __forceinline__ const ContactSeg& seg_of(const ContactLaunch& cl, int rec)
{
  int s = 0;
  if (KIND == 0)
    while (s + 1 < cl.count && rec >= cl.seg[s + 1].rec_off) s++;
  return cl.seg[s];
}

// One pair as particle i sees it (row entry e): force and moment on it.  The law
// is evaluated in the pair's own orientation (lower id first), so both particles
// compute the same bits; the first one keeps the shear history.  KIND: the
// launch's only group (ESP_SEG_*), or 0 for any mix of groups.
template <int KIND>
__device__ __forceinline__ void pair_share(const PView& p, const ContactLaunch& cl, int2 e,
                                           const double4& Pi, const double4& Vi, const double4& Ai,
                                           dv3& f, dv3& m)
{
  const bool second = e.x < 0;
  const int j = e.x & 0x7fffffff;
  const ContactSeg& g = seg_of<KIND>(cl, e.y);
  const int kind = KIND ? KIND : g.kind;
  const int c = e.y - g.rec_off;
  const double4 Pj = p.pos[j];
  const double4 P1 = second ? Pj : Pi, P2 = x_image(P1, second ? Pi : Pj, cl.period);
  const dv3 D = sub3(xyz(P1), xyz(P2));
  const double eq = P1.w + P2.w;
  if (kind == ESP_SEG_NROT_ELASTIC) {  // ElasticInteraction.cpp:54-71
    double dist = dot3(D, D);
    if (!(dist < (eq * eq))) return;
    const double kk = esp_elastic_k(g.k, g.scaling, P1.w, P2.w, cl.do2d);
    dist = sqrt(dist);
    const dv3 force = mul3(D, kk * (dist - eq) / dist);
    f = second ? force : neg3(force);
  } else if (kind == ESP_SEG_ROT_ELASTIC) {  // RotElasticInteraction.cpp:69-88
    const double rbNorm = norm3(D);
    if (!(rbNorm < eq)) return;
    const dv3 delta_r = div3(mul3(D, rbNorm - eq), rbNorm);
    const dv3 force = mul3(delta_r, esp_rotelastic_k(g.k, g.scaling, P1.w, P2.w, cl.do2d));
    f = second ? force : neg3(force);
  } else {  // RotFricInteraction.cpp:103-231
    const double4 Vj = p.vel[j], Wj = p.ang[j], st = g.ff[c];
    const double4 V1 = second ? Vj : Vi, V2 = second ? Vi : Vj;
    const double4 W1 = second ? Wj : Ai, W2 = second ? Ai : Wj;
    double kk, kks;
    esp_friction_k(g.k, g.ks, g.scaling, g.meanR, P1.w, P2.w, cl.do2d, kk, kks);
    dv3 ffr = mk3(st.x, st.y, st.z);
    bool slipping = (((int)st.w) & 1) != 0;
    dv3 f1, m1, m2;
    if (KIND == 0 && g.rigid)
      esp_rot_friction_rigid_law(xyz(P1), xyz(V1), xyz(W1), P1.w, xyz(P2), xyz(V2), xyz(W2), P2.w,
                                 kk, kks, g.mu_d, g.mu_s, cl.dt, (((int)st.w) & 2) != 0, ffr,
                                 slipping, f1, m1, m2);
    else
      esp_rot_friction_law(xyz(P1), xyz(V1), xyz(W1), P1.w, xyz(P2), xyz(V2), xyz(W2), P2.w, kk,
                           kks, g.mu_d, g.mu_s, cl.dt, ffr, slipping, f1, m1, m2);
    if (!second) g.ff_out[c] = make_double4(ffr.x, ffr.y, ffr.z, (double)((slipping ? 1 : 0) | 2));
    f = second ? neg3(f1) : f1;
    m = second ? m2 : m1;
  }
}

// The end of a wave's step: whether a particle moved beyond verletDist/2, and the
// wall forces on its 64 particles (flags fl, state before the step P) in a
// fixed-order sum; waves without candidates are not in the list the sums are
// taken over (all: there is no list, they leave zeros).
template <bool EXTRA>
__device__ __forceinline__ void step_tail(const StepCtl& ctl, const GatherParams& gp, int i, bool act,
                                          unsigned fl, double4 P, unsigned long long md,
                                          bool all = false)
{
  const int lane = threadIdx.x & 63;
  if (__ballot(md > ctl.thresh)) {
    md = wave_max_u64(md);
    if (lane == 0) atomicMax(&ctl.cur->maxdisp2, md);
  }
  if (gp.nwg > 0 && __ballot(act)) {
    double* q = gp.wall_part + (size_t)(i >> 6) * gp.nwg * 3;
    if (!__ballot(act && ((fl >> PF_WALL_SHIFT) & 0xFFu) != 0u)) {
      if (all && lane < 3 * gp.nwg) q[lane] = 0.0;
      return;
    }
    for (int w = 0; w < gp.nwg; w++) {
      const dv3 sh = act ? wall_share<EXTRA>(gp, w, i, fl, xyz(P), P.w) : mk3(0.0, 0.0, 0.0);
      const dv3 tot = mk3(wave_sum(sh.x), wave_sum(sh.y), wave_sum(sh.z));
      if (lane == 0) put3(q + 3 * w, tot);
    }
  }
}

// Blocks go round-robin to the 8 XCDs: block b's place when each XCD takes a
// contiguous range (a bijection on [0, nb)), so that neighbours' state is
// fetched into one L2
__device__ __forceinline__ int xcd_block(int b, int nb)
{
  const int d = b & 7, q8 = nb >> 3, r8 = nb & 7;
  return d * q8 + min(d, r8) + (b >> 3);
}

// One whole step of an engine without bonded groups (their laws are two orders
// of magnitude cheaper than a bond's): every particle evaluates its own pairs,
// so each pair is evaluated twice and nothing is handed from particle to
// particle through memory.  Against force slots written by one launch and
// summed by a second, a touching friction pair saves two 48-byte slots written
// and read, their two indices and activity bytes, and the step one launch.
// Positions, velocities and angular velocities are stepped into a second set of
// arrays (neighbours still read the old ones); the host swaps the sets.
//
// G lanes share a particle's pairs (row entries k = lane, lane + G, ...), their
// shares are added in row order, then one lane per particle integrates.  Bound by
// the chain row -> entry -> neighbour's position while the chip is not full: 10,000
// settling spheres 14.9 us (4.8 + 10.1 in two launches) -> 7.6, by HIP events of the
// steps that completed (a launch queued past a halt returns at once, after 1.0 us).
template <bool EXTRA, int G>
__global__ __launch_bounds__(BS) void k_contact_step(StepCtl ctl, PView p, ContactLaunch cl,
                                                     GatherParams gp)
{
  constexpr int PB = BS / G;  // particles per block
  __shared__ double acc[3 * PB];
  double none[3][3];
  const int t = threadIdx.x;
  const int p0 = xcd_block(blockIdx.x, gridDim.x) * PB;
  const int i = p0 + t;  // the particle this lane integrates (t < PB)
  const bool act = t < PB && i < p.n;
  const int pi = p0 + t / G, sub = t % G;  // the particle whose pairs it evaluates
  const int pc = pi < p.n ? pi : 0;
  const int ii = act ? i : 0;
  // loads that do not depend on others, together
  const double4 Pi = p.pos[pc];
  const unsigned fpi = p.flags[pc];
  const double mass = p.old[pc].w;
  const int a = cl.off[pc];
  const int cnt = pi < p.n ? cl.off[pc + 1] - a : 0;
  if (step_skip(ctl)) return;  // the same for the whole block
  // entries of this lane: the pair at hand, the next one and the one after it, so
  // that the next neighbour's position is on its way during a law
  int2 e0 = make_int2(0, 0), e1 = e0;
  if (sub < cnt) e0 = cl.ent[a + sub];
  if (G + sub < cnt) e1 = cl.ent[a + G + sub];
  const ContactSeg& g = cl.seg[0];
  dv3 F = wall_body_force<false, EXTRA>(gp, pc, fpi, xyz(Pi), Pi.w, mass, none);
  double4 Pj = Pi;
  if (sub < cnt) Pj = p.pos[e0.x & 0x7fffffff];
#pragma unroll 1
  for (int k = sub; k - sub < cnt; k += G) {  // as often for the G lanes of a particle
    double4 Pn = Pj;
    int2 e2 = e1;
    if (k + G < cnt) Pn = p.pos[e1.x & 0x7fffffff];
    if (k + 2 * G < cnt) e2 = cl.ent[a + k + 2 * G];
    dv3 f = mk3(0.0, 0.0, 0.0);
    if (k < cnt) {  // CElasticInteraction::calcForces (ElasticInteraction.cpp:54-71)
      const bool second = e0.x < 0;
      const double4 P1 = second ? Pj : Pi;
      const double4 P2 = x_image(P1, second ? Pi : Pj, cl.period);
      const dv3 D = sub3(xyz(P1), xyz(P2));
      double dist = dot3(D, D);
      const double eq = P1.w + P2.w;
      if (dist < (eq * eq)) {
        const double kk = esp_elastic_k(g.k, g.scaling, P1.w, P2.w, cl.do2d);
        dist = sqrt(dist);
        const dv3 force = mul3(D, kk * (dist - eq) / dist);
        f = second ? force : neg3(force);
      }
    }
    // adding the zero share of a pair apart changes no sum
#pragma unroll
    for (int q = 0; q < G; q++)
      F = add3(F, mk3(group_value<G>(f.x, q), group_value<G>(f.y, q), group_value<G>(f.z, q)));
    e0 = e1;
    e1 = e2;
    Pj = Pn;
  }
  if (sub == 0) put3(acc + 3 * (t / G), F);
  // what the integrating lanes need, on its way meanwhile
  double4 P = Pi, V = Pi, O = Pi, A = make_double4(0.0, 0.0, 0.0, 0.0), Q = A;
  unsigned fl = 0u;
  if (t < PB) {
    P = p.pos[ii];
    fl = p.flags[ii];
    V = p.vel[ii];
    O = p.old[ii];
    if (gp.rot) {
      A = p.ang[ii];
      Q = p.quat[ii];
    }
  }
  __syncthreads();
  if (t >= PB) return;
  unsigned long long md = 0;
  if (act) {
    PView po = p;
    po.pos = cl.pos_o;
    po.vel = cl.vel_o;
    po.ang = cl.ang_o;
    const dv3 F1 = mk3(acc[3 * t], acc[3 * t + 1], acc[3 * t + 2]), M1 = mk3(0.0, 0.0, 0.0);
    md = (unsigned long long)__double_as_longlong(
        damp_and_integrate<false, EXTRA>(po, gp, i, fl, F1, M1, P, V, O, A, Q, none));
  }
  step_tail<EXTRA>(ctl, gp, i, act, fl, P, md);
}

// The same step for laws with more work than an elastic contact: a block owns 64
// particles and the run of CSR entries of their pairs.  All 256 threads test the
// entries for contact; the touching ones are packed in entry order, so that the
// law runs on full waves (of the 7.5 entries a particle has in a sheared bed
// about 60 % touch, and a wave that walks its particles' runs waits for the
// longest of 64), their shares go to LDS, and the first wave adds them in entry
// order and integrates.  Bound by the latency of the gathers of the touching neighbours
// (160 bytes each, twice a pair) at the three waves a SIMD its registers allow: 616 MB
// move in a step of 1,000,000 particles, 2.5 TB/s.  Sheared bed, us a step: 30,000
// particles 17.2 (7.1 + 10.0 in two launches) -> 14.2, 1,000,000 266 -> 242; four lanes
// walking a particle's run took 20 and 252.
template <bool EXTRA, int KIND>
__global__ __launch_bounds__(BS, KIND ? 3 : 2) void k_contact_block(StepCtl ctl, PView p, ContactLaunch cl,
                                                         GatherParams gp)
{
  constexpr int PB = 64;   // particles
  constexpr int CH = 512;  // entries tested at a time
  constexpr int SC = 320;  // touching entries whose laws are evaluated at a time
  constexpr int U = CH / BS;
  __shared__ double4 sP[PB], sV[PB], sO[PB], sA[PB], sQ[PB];
  __shared__ int sOff[PB + 1];
  __shared__ double slot[6 * SC];  // [component][touching entry]
  __shared__ double sum[6 * PB];   // [component][particle]
  __shared__ int2 sEnt[CH];
  __shared__ unsigned char owner[CH];
  __shared__ unsigned short queue[CH];  // touching entries of the chunk, in order
  __shared__ unsigned long long touch_mask[CH / 64];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int p0 = xcd_block(blockIdx.x, gridDim.x) * PB;
  const int np = min(PB, p.n - p0);
  const int i = p0 + lane;  // the particle this lane loads, and in wave 0 integrates
  const int ic = lane < np ? i : p0;
  unsigned fl = 0u;
  if (wv == 0) {
    sP[lane] = p.pos[ic];
    fl = p.flags[ic];
  } else if (wv == 1) {
    sO[lane] = p.old[ic];
    sOff[lane] = cl.off[min(i, p.n)];
    if (lane == 0) sOff[PB] = cl.off[min(p0 + PB, p.n)];
  } else if (wv == 2) {
    sV[lane] = p.vel[ic];
  } else if (gp.rot) {
    sA[lane] = p.ang[ic];
    sQ[lane] = p.quat[ic];
  }
  if (step_skip(ctl)) return;  // the same for the whole block
  __syncthreads();
  double none[3][3];
  if (wv == 0) {  // the sums start from the walls' and body forces
    const dv3 F = wall_body_force<false, EXTRA>(gp, ic, fl, xyz(sP[lane]), sP[lane].w, sO[lane].w, none);
    sum[lane] = F.x;
    sum[PB + lane] = F.y;
    sum[2 * PB + lane] = F.z;
    for (int c = 3; c < 6; c++) sum[c * PB + lane] = 0.0;
  }
  const int pl = t >> 2;  // the particle whose entries and sums this thread looks after
  const int a0 = sOff[pl], a1 = sOff[pl + 1];
  const int E0 = sOff[0], E1 = sOff[PB];
  for (int cb = E0; cb < E1; cb += CH) {
    int2 en[U];
    double4 Pn[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = cb + u * BS + t;
      en[u] = k < E1 ? cl.ent[k] : make_int2(0, 0);
    }
    // whose entries they are: 4 threads a particle
    const int ca = max(a0, cb) - cb, ce = min(a1, cb + CH) - cb;
    for (int k = ca + (t & 3); k < ce; k += 4) owner[k] = (unsigned char)pl;
#pragma unroll
    for (int u = 0; u < U; u++)
      if (cb + u * BS + t < E1) Pn[u] = p.pos[en[u].x & 0x7fffffff];
    __syncthreads();
    bool on[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      on[u] = false;
      if (cb + u * BS + t < E1) {
        sEnt[u * BS + t] = en[u];
        const bool second = en[u].x < 0;
        const double4 Pi = sP[owner[u * BS + t]];
        const double4 P1 = second ? Pn[u] : Pi;
        const double4 P2 = x_image(P1, second ? Pi : Pn[u], cl.period);
        const dv3 D = sub3(xyz(P1), xyz(P2));
        const double eq = P1.w + P2.w;
        const ContactSeg& g = seg_of<KIND>(cl, en[u].y);
        const int kind = KIND ? KIND : g.kind;
        // (RotElastic tests |D| < eq; a pair that only rounding separates from
        // that is left to its law)
        on[u] = kind == ESP_SEG_ROT_ELASTIC ? dot3(D, D) <= (eq * eq) * 1.000001
                                            : dot3(D, D) < (eq * eq);
        if (!on[u] && !second && kind == ESP_SEG_ROT_FRICTION) clear_history(g, en[u].y - g.rec_off);
      }
      const unsigned long long m = __ballot(on[u]);
      if (lane == 0) touch_mask[u * (BS / 64) + wv] = m;
    }
    __syncthreads();
    // touching entries before entry x of the chunk: lane k of every wave holds
    // those before the k-th 64 (every lane calls it)
    int before = 0;
    {
      const int pc = lane < CH / 64 ? __popcll(touch_mask[lane]) : 0;
      int inc = pc;
#pragma unroll
      for (int d = 1; d < 16; d <<= 1) {
        const int v = __shfl_up(inc, d, 64);
        if (lane >= d) inc += v;
      }
      before = inc - pc;
    }
    auto rank = [&](int x) {
      const int w = x >> 6;
      const unsigned long long m = w < CH / 64 ? touch_mask[w] : 0ull;
      return __shfl(before, w, 64) + __popcll(m & ((1ull << (x & 63)) - 1ull));
    };
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int q = rank(u * BS + t);
      if (on[u]) queue[q] = (unsigned short)(u * BS + t);
    }
    const int nq = rank(CH);
    const int qa = rank(min(ca, CH)), qe = rank(max(ce, 0));
    __syncthreads();
    for (int qb = 0; qb < nq; qb += SC) {
      const int qn = min(nq - qb, SC);
#pragma unroll 1
      for (int q = t; q < qn; q += BS) {
        const int x = queue[qb + q];
        const int2 e = sEnt[x];
        const int o = owner[x];
        dv3 f = mk3(0.0, 0.0, 0.0), m = f;
        pair_share<KIND>(p, cl, e, sP[o], sV[o], sA[o], f, m);
        slot[q] = f.x;
        slot[SC + q] = f.y;
        slot[2 * SC + q] = f.z;
        slot[3 * SC + q] = m.x;
        slot[4 * SC + q] = m.y;
        slot[5 * SC + q] = m.z;
      }
      __syncthreads();
      // each particle's shares in entry order; its 4 threads take the components
      // (force x, y, z and moment x; moment y, z)
      {
        const int u0 = max(qa, qb) - qb, u1 = min(qe, qb + SC) - qb;
        const int c = t & 3;
        if (u0 < u1) {
          double s0 = sum[c * PB + pl], s1 = c < 2 ? sum[(c + 4) * PB + pl] : 0.0;
          for (int q = u0; q < u1; q++) {
            s0 = s0 + slot[c * SC + q];
            if (c < 2) s1 = s1 + slot[(c + 4) * SC + q];
          }
          sum[c * PB + pl] = s0;
          if (c < 2) sum[(c + 4) * PB + pl] = s1;
        }
      }
      __syncthreads();
    }
  }
  if (wv != 0) return;
  const bool act = lane < np;
  const double4 P = sP[lane];
  unsigned long long md = 0;
  if (act) {
    PView po = p;
    po.pos = cl.pos_o;
    po.vel = cl.vel_o;
    po.ang = cl.ang_o;
    const dv3 F = mk3(sum[lane], sum[PB + lane], sum[2 * PB + lane]);
    const dv3 M = mk3(sum[3 * PB + lane], sum[4 * PB + lane], sum[5 * PB + lane]);
    md = (unsigned long long)__double_as_longlong(damp_and_integrate<false, EXTRA>(
        po, gp, i, fl, F, M, P, sV[lane], sO[lane], sA[lane], sQ[lane], none));
  }
  step_tail<EXTRA>(ctl, gp, i, act, fl, P, md);
}

// The gather for 6-double slots: four lanes share a particle's slots.  A
// block is 64 particles.  The activity bytes of a run come in as aligned words,
// one a lane, 64 slots at a time, and become one bit mask that all four lanes
// hold; each lane then loads every fourth active slot, and the shares are added
// in slot order.  One lane for each of the particles (the first wave) integrates;
// its state is on its way meanwhile.
// With one lane a particle the run's words, then up to eight slots of 48 bytes,
// were a chain in every lane: 9.0 us for 2,000 particles (13 us where flagged
// pairs make runs of 200 slots), 15.4 us for 100,000.  RQ: active slots a lane has
// in flight, as a turn of the sum waits for memory once.  One / three: 7.1 / 6.8 us
// for 2,000 particles, 9.1 / 7.9 for 5,000 with flagged pairs, 8.4 / 8.1 for 30,000,
// but 11.1 / 12.7 for 60,000, where the registers of three cost a wave a SIMD:
// three up to GATHER_DEEP.
template <bool EXTRA, int RQ>
__global__ __launch_bounds__(BS) void k_gather_integrate(StepCtl ctl, PView p, GatherParams gp)
{
  constexpr int G = 4, PB = BS / G;
  __shared__ double sum[6 * PB];
  double none[3][3];
  const int t = threadIdx.x;
  const int p0 = xcd_block(blockIdx.x, gridDim.x) * PB;
  const int pi = p0 + t / G, sub = t % G;  // the particle whose slots it adds
  const int pc = pi < p.n ? pi : 0;
  const int i = p0 + t;  // the particle it integrates (t < PB)
  const bool act = t < PB && i < p.n;
  const int ii = act ? i : 0;
  const int e0 = gp.inc_off[pc], e1 = gp.inc_off[pc + 1], xcnt = gp.xcnt[pc];
  double4 P = make_double4(0.0, 0.0, 0.0, 0.0), V = P, O = P, A = P, Q = P;
  unsigned fl = 0u;
  if (t < PB) {
    P = p.pos[ii];
    fl = p.flags[ii];
    V = p.vel[ii];
    O = p.old[ii];
    if (gp.rot) {
      A = p.ang[ii];
      Q = p.quat[ii];
    }
  }
  const unsigned* sw = reinterpret_cast<const unsigned*>(gp.sact);
  const int nmain = pi < p.n ? e1 - e0 : 0;
  const int nx = pi < p.n ? xcnt : 0;
  const int w0 = e0 >> 2, sh = e0 & 3;  // the run starts sh bytes into word w0
  // words of the first 64 slots, and the appendix's activity
  unsigned wd[4];
#pragma unroll
  for (int r = 0; r < 4; r++) wd[r] = 16 * r + 4 * sub < sh + nmain ? sw[w0 + 4 * r + sub] : 0u;
  const unsigned ax = sub < nx ? gp.sact[gp.xbase + ESP_XSLOTS * pc + sub] : 0u;
  if (step_skip(ctl)) return;  // the same for the whole block
  // pairs appended by this step's incremental update are covered by the force
  // blocks from the next step on
  if (gp.n_app && blockIdx.x == 0 && t == 0) gp.n_app[1] = gp.n_app[0];
  if (t < PB) {
    if (act && gp.nwg > 0 && ctl.guarded && ctl.prev->nbroken > 0) {
      // bonds broke in the previous step: the reference's updateInteractions
      // re-Updates the wall groups (EWallInteractionGroup.hpp:57-82) before forces
      fl = wall_membership(gp.grid, gp.nwg, gp.wall, P, fl);
      p.flags[i] = fl;
    }
    const dv3 F = wall_body_force<false, EXTRA>(gp, ii, act ? fl : 0u, xyz(P), P.w, O.w, none);
    put3(sum + 6 * t, F);
  }
  __syncthreads();
  const double* s0 = sum + 6 * (t / G);
  dv3 F = mk3(s0[0], s0[1], s0[2]), M = mk3(0.0, 0.0, 0.0);
  auto add_active = [&](unsigned long long m, size_t base) {
    for (int k = 0; k < sub; k++) m &= m - 1ull;  // this lane's first
    while (__ballot(m != 0ull)) {
      double v[RQ][6];
#pragma unroll
      for (int r = 0; r < RQ; r++) {
        double2 qa = make_double2(0.0, 0.0), qb = qa, qc = qa;
        if (m) {
          const double2* q =
              reinterpret_cast<const double2*>(gp.slots + 6 * (base + __builtin_ctzll(m)));
          qa = q[0];
          qb = q[1];
          qc = q[2];
          for (int k = 0; k < G; k++) m &= m - 1ull;
        }
        v[r][0] = qa.x; v[r][1] = qa.y; v[r][2] = qb.x;
        v[r][3] = qb.y; v[r][4] = qc.x; v[r][5] = qc.y;
      }
#pragma unroll
      for (int r = 0; r < RQ; r++)
#pragma unroll
        for (int k = 0; k < G; k++) {
          F = add3(F, mk3(group_value<G>(v[r][0], k), group_value<G>(v[r][1], k),
                          group_value<G>(v[r][2], k)));
          M = add3(M, mk3(group_value<G>(v[r][3], k), group_value<G>(v[r][4], k),
                          group_value<G>(v[r][5], k)));
        }
    }
  };
  // 64 bytes of activity a turn, from the run's first aligned word
  for (int b = 0; __ballot(b < sh + nmain); b += 64) {
    unsigned long long m = 0ull;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const unsigned v = wd[r];
      const unsigned m4 = (v & 1u) | ((v >> 7) & 2u) | ((v >> 14) & 4u) | ((v >> 21) & 8u);
      m |= (unsigned long long)m4 << (16 * r + 4 * sub);
      const int nb = b + 64 + 16 * r + 4 * sub;
      wd[r] = nb < sh + nmain ? sw[w0 + (nb >> 2)] : 0u;
    }
    m = group_or(m);
    const int lo = b == 0 ? sh : 0, hi = min(64, sh + nmain - b);
    if (hi <= lo) m = 0ull;
    else m &= (hi == 64 ? ~0ull : ((1ull << hi) - 1ull)) & (~0ull << lo);
    add_active(m, (size_t)(4ll * w0 + b));
  }
  if (__ballot(nx > 0)) {
    const unsigned long long m = group_or((unsigned long long)(ax ? 1u : 0u) << sub);
    add_active(m, (size_t)gp.xbase + (size_t)ESP_XSLOTS * pc);
  }
  __syncthreads();  // the walls' forces have been read
  if (sub == 0) {
    double* o = sum + 6 * (t / G);
    put3(o, F);
    put3(o + 3, M);
  }
  __syncthreads();
  if (t >= PB) return;
  unsigned long long md = 0;
  if (act) {
    const double* o = sum + 6 * t;
    md = (unsigned long long)__double_as_longlong(
        damp_and_integrate<false, EXTRA>(p, gp, i, fl, mk3(o[0], o[1], o[2]), mk3(o[3], o[4], o[5]), P,
                                         V, O, A, Q, none));
  }
  step_tail<EXTRA>(ctl, gp, i, act, fl, P, md, true);
}

// The same with one lane a particle, for particle counts that fill the chip by
// themselves (four lanes then only add waves: 66 us against 80 us for 600,000
// particles, equal at 100,000).  A run's activity bytes become a bit mask in one
// round of loads, GATHER_WIN slots at a time, and the active slots load
// GATHER_CHUNK together.
template <bool EXTRA>
__global__ __launch_bounds__(BS) void k_gather_wide(StepCtl ctl, PView p, GatherParams gp)
{
  constexpr int GATHER_CHUNK = 8;  // active slots fetched together
  constexpr int GATHER_WIN = 28;   // slots per activity-mask window (8 words with any offset)
  static_assert(GATHER_WIN < 32 && GATHER_WIN % 4 == 0, "a window's mask fits 32 bits");
  double none[3][3];
  if (step_skip(ctl)) return;
  if (gp.n_app && blockIdx.x == 0 && threadIdx.x == 0) gp.n_app[1] = gp.n_app[0];
  const int i = blockIdx.x * BS + threadIdx.x;
  const bool act = i < p.n;
  const int ii = act ? i : 0;
  // every load that does not depend on another is issued here, together
  const double4 P = p.pos[ii];
  unsigned fl = p.flags[ii];
  const double4 V = p.vel[ii];
  const double4 O = p.old[ii];
  const int e0 = gp.inc_off[ii], e1 = gp.inc_off[ii + 1];
  const int xcnt = gp.xcnt[ii];
  double4 A = make_double4(0.0, 0.0, 0.0, 0.0), Q = A;
  if (gp.rot) {
    A = p.ang[ii];
    Q = p.quat[ii];
  }
  if (act && gp.nwg > 0 && ctl.guarded && ctl.prev->nbroken > 0) {
    // as in k_gather_integrate
    fl = wall_membership(gp.grid, gp.nwg, gp.wall, P, fl);
    p.flags[i] = fl;
  }
  unsigned long long md = 0;
  if (act) {
    dv3 F = wall_body_force<false, EXTRA>(gp, i, fl, xyz(P), P.w, O.w, none);
    dv3 M = mk3(0.0, 0.0, 0.0);
    const int nmain = e1 - e0;
    const int cnt = nmain + xcnt;
    const unsigned* sw = reinterpret_cast<const unsigned*>(gp.sact);
    for (int wb = 0; wb < cnt; wb += GATHER_WIN) {
      unsigned mask = 0;
      int base = 0;  // slot index of mask bit 0
      if (wb < nmain) {
        const int s0 = e0 + wb, nw = min(GATHER_WIN, nmain - wb), sh = s0 & 3;
        unsigned wv[GATHER_WIN / 4 + 1];
#pragma unroll
        for (int k = 0; k <= GATHER_WIN / 4; k++) wv[k] = 4 * k < sh + nw ? sw[(s0 >> 2) + k] : 0u;
        unsigned long long m = 0;
#pragma unroll
        for (int k = 0; k <= GATHER_WIN / 4; k++) {
          const unsigned v = wv[k];
          const unsigned long long m4 = (v & 1u) | ((v >> 7) & 2u) | ((v >> 14) & 4u) | ((v >> 21) & 8u);
          m |= m4 << (4 * k);
        }
        mask = (unsigned)(m >> sh) & ((1u << nw) - 1u);  // nw <= GATHER_WIN < 32
        base = s0;
      } else {
        // the appendix slots follow the run (at most ESP_XSLOTS of them)
        for (int t = 0; t < xcnt; t++)
          if (gp.sact[gp.xbase + ESP_XSLOTS * i + t]) mask |= 1u << t;
        base = gp.xbase + ESP_XSLOTS * i;
      }
      while (mask) {
        double2 qa[GATHER_CHUNK], qb[GATHER_CHUNK], qc[GATHER_CHUNK];
        int sl[GATHER_CHUNK];
        bool on[GATHER_CHUNK];
#pragma unroll
        for (int k = 0; k < GATHER_CHUNK; k++) {
          on[k] = mask != 0;
          sl[k] = base + (on[k] ? __builtin_ctz(mask) : 0);
          mask &= mask - 1u;
        }
#pragma unroll
        for (int k = 0; k < GATHER_CHUNK; k++) {
          if (on[k]) {
            const double2* q = reinterpret_cast<const double2*>(gp.slots + 6 * (size_t)sl[k]);
            qa[k] = q[0];
            qb[k] = q[1];
            qc[k] = q[2];
          }
        }
#pragma unroll
        for (int k = 0; k < GATHER_CHUNK; k++) {
          if (!on[k]) continue;
          F = add3(F, mk3(qa[k].x, qa[k].y, qb[k].x));
          M = add3(M, mk3(qb[k].y, qc[k].x, qc[k].y));
        }
      }
      // the appendix starts its own window right after the run
      if (wb < nmain && wb + GATHER_WIN >= nmain) wb = nmain - GATHER_WIN;
    }
    md = (unsigned long long)__double_as_longlong(
        damp_and_integrate<false, EXTRA>(p, gp, i, fl, F, M, P, V, O, A, Q, none));
  }
  step_tail<EXTRA>(ctl, gp, i, act, fl, P, md, true);
}

// the 64-particle groups holding wall candidates, ascending (one block; marks
// from k_wall_update)
__global__ __launch_bounds__(1024) void k_wall_list(int ng, const int* mark, int* list, int* list_n)
{
  __shared__ int wsum[16], base_s;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  int base = 0;
  for (int b0 = 0; b0 < ng; b0 += 1024) {
    const bool on = b0 + t < ng && mark[b0 + t] != 0;
    const unsigned long long bal = __ballot(on);
    if (lane == 0) wsum[wv] = __popcll(bal);
    __syncthreads();
    int pre = base;
    for (int w = 0; w < wv; w++) pre += wsum[w];
    if (on) list[pre + __popcll(bal & ((1ull << lane) - 1ull))] = b0 + t;
    if (t == 1023) base_s = pre + __popcll(bal);
    __syncthreads();
    base = base_s;
  }
  if (t == 0) *list_n = base;
}

// ---------------------------------------------------------------------------
// neighbour table
// ---------------------------------------------------------------------------
__global__ void k_cells_count(PView p, GridParams g, int* cell, int* cell_count, int* n_out)
{
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i >= p.n) return;
  const double4 P = p.pos[i];
  int ix, iy, iz, c = -1;
  if (cell_coords(g, P.x, P.y, P.z, ix, iy, iz) && ix >= 0 && ix < g.nx && iy >= 0 && iy < g.ny &&
      iz >= 0 && iz < g.nz)
    c = g.ny * g.nz * ix + g.nz * iy + iz;
  cell[i] = c;
  if (c < 0) atomicAdd(n_out, 1);
  else atomicAdd(&cell_count[c], 1);
  // resetDisplacement (Particle.h:124)
  const double4 O = p.old[i];
  p.old[i] = make_double4(P.x, P.y, P.z, O.w);
}

__global__ void k_cells_fill(int n, const int* cell, const int* cell_start, int* cell_fill,
                             int* cell_items)
{
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i >= n) return;
  const int c = cell[i];
  if (c < 0) return;
  const int k = atomicAdd(&cell_fill[c], 1);
  cell_items[cell_start[c] + k] = i;
}

// cell contents in particle-array order
__global__ void k_cells_sort(int ncell, const int* cell_start, int* items)
{
  const int c = blockIdx.x * BS + threadIdx.x;
  if (c >= ncell) return;
  const int a = cell_start[c], b = cell_start[c + 1];
  for (int i = a + 1; i < b; i++) {
    const int v = items[i];
    int j = i - 1;
    while (j >= a && items[j] > v) {
      items[j + 1] = items[j];
      j--;
    }
    items[j + 1] = v;
  }
}


// Pairs of particle p with every particle q of higher id in the 27 cells around
// p's cell: the full list keeps pairs with |x_p - x_q|^2 <= (r_p + r_q + alpha)^2
// (ntable.hpp:471-521); the flagged list keeps pairs of two flagged particles
// without a distance test (ntable.hpp:532-583).  Two passes: the first counts,
// the second writes each particle's run in the order of the partner's slot.
//
// 32 lanes search for one particle, a cell each (a single lane's chain of 27
// cells took 53.5 us a launch for 10,000 particles, all of it latency: 6.5 us so);
// the second pass collects a particle's partners in LDS and places each by counting
// the smaller ones.  Runs longer than PAIRS_CAP (wide size ranges, flagged lists)
// are merged from the cells' own orders by binary searches: counting costs the
// square of the run, which is small up to PAIRS_CAP and was 142 ms a search for a
// large sphere under 1,000 small ones (15 ms so, most of it sorting their cells).
#define PAIRS_CAP 192
template <bool EMIT, bool FLAGGED>
__global__ __launch_bounds__(BS) void k_pairs(PView p, GridParams g, double alpha, const int* cell,
                                              const int* cell_start, const int* cell_items, int* cnt,
                                              const int* off, int cap, int* out_p, int* out_q,
                                              long long* out_key)
{
  constexpr int L = 32, PPB = BS / L;
  __shared__ int list[EMIT ? PPB * PAIRS_CAP : 1];
  __shared__ int num[PPB];
  const int grp = threadIdx.x / L, l = threadIdx.x % L;
  const int pi = blockIdx.x * PPB + grp;
  const bool on = pi < p.n && (!FLAGGED || (p.flags[pi] & PF_FLAG));
  if (l == 0) num[grp] = 0;
  __syncthreads();
  int c2 = -1;  // this lane's cell
  double4 P = make_double4(0.0, 0.0, 0.0, 0.0);
  int idp = 0;
  if (on && l < 27) {
    const int c = cell[pi];
    P = p.pos[pi];
    idp = p.id[pi];
    const int cx = c / (g.ny * g.nz);
    const int rem = c - cx * (g.ny * g.nz);
    const int cy = rem / g.nz;
    int x = cx + l / 9 - 1;
    const int y = cy + (l / 3) % 3 - 1, z = rem - cy * g.nz + l % 3 - 1;
    // circular x: the stencil wraps (nx >= 3, so its cells are distinct)
    if (g.circ_x) x = (x + g.nx) % g.nx;
    if (x >= 0 && x < g.nx && y >= 0 && y < g.ny && z >= 0 && z < g.nz)
      c2 = g.ny * g.nz * x + g.nz * y + z;
  }
  auto taken = [&](int q) {
    if (p.id[q] <= idp) return false;
    if (FLAGGED) return (p.flags[q] & PF_FLAG) != 0u;
    const double4 Q = x_image(P, p.pos[q], g.period);
    const dv3 d = sub3(xyz(P), xyz(Q));
    const double dist2 = dot3(d, d);
    const double dmax = P.w + Q.w + alpha;
    return dist2 <= (dmax * dmax);
  };
  int count = 0;
  if (c2 >= 0) {
    const int t1 = cell_start[c2 + 1];
    for (int t = cell_start[c2]; t < t1; t++) {
      const int q = cell_items[t];
      if (!taken(q)) continue;
      count++;
      if (EMIT) {
        const int k = atomicAdd(&num[grp], 1);
        if (k < PAIRS_CAP) list[grp * PAIRS_CAP + k] = q;
      }
    }
  }
  if (!EMIT) {
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) count += __shfl_xor(count, o, L);
    if (l == 0 && pi < p.n) cnt[pi] = count;
    return;
  }
  __syncthreads();
  const int m = num[grp];
  if (!on || m == 0) return;
  const int base = off[pi];
  auto put = [&](int q, int r) {
    if (base + r >= cap) return;  // the caller sees the total and comes back with room
    out_p[base + r] = pi;
    out_q[base + r] = q;
    out_key[base + r] = pair_key(pi, q);
  };
  const int* mine = list + grp * PAIRS_CAP;
  if (m <= PAIRS_CAP) {
    for (int e = l; e < m; e += L) {
      const int q = mine[e];
      int r = 0;
      for (int k = 0; k < m; k++) r += mine[k] < q ? 1 : 0;
      put(q, r);
    }
  } else if (base + m > cap) {
    // no room for the run: what of it fits only has to name particles
    for (int r = l; r < m; r += L) put(pi, r);
  } else {
    // The cells list their particles in slot order, so the partners of a cell are a
    // sorted segment (out_q), and a partner's place is the sum of its places in the
    // 27 segments; (partner, place) goes through out_key, since out_q is read until
    // every place is known.  The group's lanes are in one wave: a fence orders them.
    int* seg = list + grp * PAIRS_CAP;  // the segments' starts
    int before = count;
#pragma unroll
    for (int o = 1; o < L; o <<= 1) {
      const int u = __shfl_up(before, o, L);
      if (l >= o) before += u;
    }
    before -= count;
    if (l < 28) seg[l] = base + before;  // lanes past the cells: the end
    if (c2 >= 0) {
      int w = base + before;
      const int t1 = cell_start[c2 + 1];
      for (int t = cell_start[c2]; t < t1; t++)
        if (taken(cell_items[t])) out_q[w++] = cell_items[t];
    }
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
    for (int e = base + l; e < base + m; e += L) {
      const int q = out_q[e];
      int r = 0;
      for (int k = 0; k < 27; k++) {
        const int s0 = seg[k];
        int lo = s0, hi = seg[k + 1];
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (out_q[mid] < q) lo = mid + 1;
          else hi = mid;
        }
        r += lo - s0;
      }
      out_key[e] = ((long long)q << 32) | (long long)r;
    }
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
    for (int e = base + l; e < base + m; e += L) {
      const long long v = out_key[e];
      out_q[base + (int)(v & 0xffffffffll)] = (int)(v >> 32);
      out_p[e] = pi;
    }
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
    for (int e = base + l; e < base + m; e += L) out_key[e] = pair_key(pi, out_q[e]);
  }
}

// ---------------------------------------------------------------------------
// erasure of particles outside the padded grid (NeighborTable::build,
// ntable.hpp:281-286): stable compaction in slot order
// ---------------------------------------------------------------------------
__global__ void k_keep_cells(int n, const int* cell, int* keep)
{
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i < n) keep[i] = cell[i] >= 0 ? 1 : 0;
}

// new slot of every particle, -1 for an erased one
__global__ void k_new_slot(int n, const int* keep, const int* off, int* nslot)
{
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i < n) nslot[i] = keep[i] ? off[i] : -1;
}

template <class T>
__global__ void k_compact_field(int n, int width, const int* keep, const int* off, const T* src,
                                T* dst)
{
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i >= n || !keep[i]) return;
  for (int c = 0; c < width; c++) dst[(size_t)width * off[i] + c] = src[(size_t)width * i + c];
}

// an interaction's particles at their new slots; kept while both survive
// (PIS_E::rebuild, pi_storage_e.hpp:111-155)
__global__ void k_remap_pairs(int nc, const int2* ij, const int* nslot, int2* out, int* keep)
{
  const int c = blockIdx.x * BS + threadIdx.x;
  if (c >= nc) return;
  const int2 e = ij[c];
  const int a = e.x >= 0 ? nslot[e.x] : -1, b = e.y >= 0 ? nslot[e.y] : -1;
  out[c] = make_int2(a, b);
  keep[c] = (a >= 0 && b >= 0) ? 1 : 0;
}

// the kept pairs of a dynamic group with their slot keys (order kept: slots
// are renumbered monotonically, so the list stays sorted by key)
__global__ void k_pack_dyn(int nc, const int* keep, const int* off, const int2* ij,
                           const double4* ff, int2* oij, long long* okey, double4* off_)
{
  const int c = blockIdx.x * BS + threadIdx.x;
  if (c >= nc || !keep[c]) return;
  const int w = off[c];
  const int2 e = ij[c];
  oij[w] = e;
  okey[w] = pair_key(e.x, e.y);
  if (off_) off_[w] = ff[c];
}

// the candidate particles of wall group w (flag bit PF_WALL_SHIFT + w): slot,
// flags, position and (bonded walls) initial position, in any order; all are
// counted, the first cap are stored
__global__ void k_wall_cands(PView p, int w, const double4* init, int cap, int* cnt, int* slot,
                             unsigned* flg, double4* pos, double4* ipos)
{
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i >= p.n) return;
  const unsigned f = p.flags[i];
  if (!((f >> (PF_WALL_SHIFT + w)) & 1u)) return;
  const int k = atomicAdd(cnt, 1);
  if (k >= cap) return;
  slot[k] = i;
  flg[k] = f;
  pos[k] = p.pos[i];
  if (init) ipos[k] = init[i];
}

// What the bonded servo's iteration needs of wall group w's candidates, in one
// pass: out[block][8] = (stiffness sum of the tagged inner ones, their force sum
// at the wall displacement disp, the least gap of the untagged inner ones to the
// wall, candidates), written to page-locked host memory and added up there in
// block order.  Waves take the 64-particle groups of list (all groups: nullptr).
__global__ __launch_bounds__(BS) void k_servo_sums(PView p, WallParam W, int w, int do2d, int ng,
                                                   const double4* init, const int* list,
                                                   const int* list_n, double* out)
{
  __shared__ double part[BS / 64][6];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = list ? *list_n : ng;
  double K = 0.0, sx = 0.0, sy = 0.0, sz = 0.0, gap = 1e300, cnt = 0.0;
  for (int t = blockIdx.x * (BS / 64) + wv; t < m; t += gridDim.x * (BS / 64)) {
    const int i = (list ? list[t] : t) * 64 + lane;
    if (i >= p.n) continue;
    const unsigned fl = p.flags[i];
    if (!((fl >> (PF_WALL_SHIFT + w)) & 1u)) continue;
    cnt = cnt + 1.0;
    if (!((fl >> (PF_INNER_SHIFT + w)) & 1u)) continue;
    const double4 P = p.pos[i];
    if ((fl >> (PF_BTAG_SHIFT + w)) & 1u) {
      const double kb = W.k * (do2d ? 1.0 : 3.1415926536 * P.w);
      const dv3 D = sub3(sub3(xyz(P), xyz(init[i])), mk3(W.disp[0], W.disp[1], W.disp[2]));
      K = K + kb;
      sx = sx + D.x * kb;
      sy = sy + D.y * kb;
      sz = sz + D.z * kb;
    } else {
      const double dist = dot3(sub3(xyz(P), mk3(W.o[0], W.o[1], W.o[2])),
                               mk3(W.nrm[0], W.nrm[1], W.nrm[2]));
      gap = fmin(gap, dist - P.w);
    }
  }
  K = wave_sum(K);
  sx = wave_sum(sx);
  sy = wave_sum(sy);
  sz = wave_sum(sz);
  cnt = wave_sum(cnt);
  for (int o = 32; o > 0; o >>= 1) gap = fmin(gap, __shfl_xor(gap, o, 64));
  if (lane == 0) {
    part[wv][0] = K;
    part[wv][1] = sx;
    part[wv][2] = sy;
    part[wv][3] = sz;
    part[wv][4] = gap;
    part[wv][5] = cnt;
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    double a = part[0][threadIdx.x];
    for (int k = 1; k < BS / 64; k++)
      a = threadIdx.x == 4 ? fmin(a, part[k][4]) : a + part[k][threadIdx.x];
    out[8 * blockIdx.x + threadIdx.x] = a;
  }
}

// a field in id order, packed: 3 or 4 components, or (width 1) the fourth alone
__global__ void k_pack_ordered(int n, const int* order, const double4* src, int width, double* out)
{
  const int k = blockIdx.x * BS + threadIdx.x;
  if (k >= n) return;
  const double4 v = src[order[k]];
  if (width == 1) {
    out[k] = v.w;
    return;
  }
  double* o = out + (size_t)width * k;
  o[0] = v.x;
  o[1] = v.y;
  o[2] = v.z;
  if (width == 4) o[3] = v.w;
}

__global__ void k_wall_mark_ordered(int no, const int* ord_slot, const unsigned* flags, int w,
                                    int* mark)
{
  const int o = blockIdx.x * BS + threadIdx.x;
  if (o >= no) return;
  const int s = ord_slot[o];
  mark[o] = (s >= 0 && ((flags[s] >> (PF_WALL_SHIFT + w)) & 1u)) ? 1 : 0;
}

__global__ void k_wall_pack_ordered(int no, const int* ord_slot, const int* mark, const int* off,
                                    PView p, const double4* init, WallCand* out)
{
  const int o = blockIdx.x * BS + threadIdx.x;
  if (o >= no || !mark[o]) return;
  const int s = ord_slot[o];
  const double4 x0 = init ? init[s] : make_double4(0.0, 0.0, 0.0, 0.0);
  WallCand& c = out[off[o]];
  c.pos = p.pos[s];
  c.ix = x0.x;
  c.iy = x0.y;
  c.iz = x0.z;
  c.flags = p.flags[s];
  c.pad = 0u;
}

__global__ void k_clear_flag_bit(PView p, UpdState* st)
{
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i < p.n) p.flags[i] &= ~PF_FLAG;
  if (i == 0) st->fcount = 0;
}

__device__ __forceinline__ int bsearch_key(const long long* a, int n, long long key)
{
  int lo = 0, hi = n - 1;
  while (lo <= hi) {
    const int mid = (lo + hi) >> 1;
    const long long v = a[mid];
    if (v == key) return mid;
    if (v < key) lo = mid + 1;
    else hi = mid - 1;
  }
  return -1;
}
// number of elements < key (strict) or <= key
__device__ __forceinline__ int lower_bound_key(const long long* a, int n, long long key)
{
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (a[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}
__device__ __forceinline__ int upper_bound_key(const long long* a, int n, long long key)
{
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (a[mid] <= key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// PIS_ED::update on a rebuilt table (pi_storage_ed.hpp:97-136): a candidate is
// kept unless excluded; it inherits the history of the stored interaction with
// the same key if that one is persistent (RotFricInteraction.cpp:345-351).
// nc_dev (nullable): the candidates there are, when only the device knows; nc is
// then the room they have, and marks beyond them are zero
__global__ void k_ed_mark(int nc, const int* nc_dev, const int* cp, const int* cq, const long long* ckey, ExclSet ex,
                          const long long* okey, int nold, const int2* oij, PView p, double period,
                          int* keep, int* src)
{
  const int c = blockIdx.x * BS + threadIdx.x;
  if (c >= nc) return;
  if (nc_dev && c >= *nc_dev) {
    keep[c] = 0;
    return;
  }
  const long long key = ckey[c];
  if (rejected(ex, pair_key(p.id[cp[c]], p.id[cq[c]]), cp[c], cq[c])) {
    keep[c] = 0;
    src[c] = -1;
    return;
  }
  keep[c] = 1;
  int s = -1;
  const int j = bsearch_key(okey, nold, key);
  if (j >= 0) {
    const int2 e = oij[j];
    const double4 P1 = p.pos[e.x], P2 = x_image(P1, p.pos[e.y], period);
    const dv3 D = sub3(xyz(P1), xyz(P2));
    const double dist = dot3(D, D);
    const double eq = P1.w + P2.w;
    if (dist <= (eq * eq)) s = j;
  }
  src[c] = s;
}

__global__ void k_ne_mark(int nc, const int* nc_dev, const int* cp, const int* cq, const int* id,
                          ExclSet ex, int* keep)
{
  const int c = blockIdx.x * BS + threadIdx.x;
  if (c >= nc) return;
  if (nc_dev && c >= *nc_dev) keep[c] = 0;
  else keep[c] = rejected(ex, pair_key(id[cp[c]], id[cq[c]]), cp[c], cq[c]) ? 0 : 1;
}

__global__ void k_pair_emit(int nc, const int* keep, const int* off, const int* cp, const int* cq,
                            const long long* ckey, const int* src, const double4* off_ff, int cap,
                            int2* nij, long long* nkey, double4* nff)
{
  const int c = blockIdx.x * BS + threadIdx.x;
  if (c >= nc || !keep[c]) return;
  const int w = off[c];
  if (w >= cap) return;  // the caller sees the total and comes back with room
  nij[w] = make_int2(cp[c], cq[c]);
  nkey[w] = ckey[c];
  if (nff) {
    const int s = src ? src[c] : -1;
    nff[w] = s >= 0 ? off_ff[s] : make_double4(0.0, 0.0, 0.0, 0.0);
  }
}

// pairs of the flagged list that a group takes: not excluded and (for history
// groups) not already stored (pi_storage_ed.hpp:137-156, pi_storage_ne.hpp:79-96)
__global__ void k_filter_new(int nc, const int* cp, const int* cq, const int* id,
                             const long long* ckey, ExclSet ex, HashRef present, int check_present,
                             int* keep)
{
  const int c = blockIdx.x * BS + threadIdx.x;
  if (c >= nc) return;
  int k = rejected(ex, pair_key(id[cp[c]], id[cq[c]]), cp[c], cq[c]) ? 0 : 1;
  if (k && check_present && hs_find(present, ckey[c]) >= 0) k = 0;
  keep[c] = k;
}

__global__ void k_pack_pairs(int n, const int* keep, const int* off, const int* cp, const int* cq,
                             const long long* ckey, int2* ij, long long* key)
{
  const int c = blockIdx.x * BS + threadIdx.x;
  if (c >= n || !keep[c]) return;
  const int w = off[c];
  ij[w] = make_int2(cp[c], cq[c]);
  key[w] = ckey[c];
}

// merge of two key-sorted lists; equal keys keep stored entries first
__global__ void k_merge(int nold, const int2* oij, const long long* okey, const double4* off_,
                        int nnew, const int2* nij_in, const long long* nkey_in,
                        const double4* nff_in, int2* ij_out, long long* key_out, double4* ff_out)
{
  const int t = blockIdx.x * BS + threadIdx.x;
  if (t < nold) {
    const long long key = okey[t];
    const int w = t + lower_bound_key(nkey_in, nnew, key);
    ij_out[w] = oij[t];
    key_out[w] = key;
    if (ff_out) ff_out[w] = off_[t];
  } else if (t < nold + nnew) {
    const int j = t - nold;
    const long long key = nkey_in[j];
    const int w = j + upper_bound_key(okey, nold, key);
    ij_out[w] = nij_in[j];
    key_out[w] = key;
    if (ff_out) ff_out[w] = nff_in ? nff_in[j] : make_double4(0.0, 0.0, 0.0, 0.0);
  }
}


__global__ void k_fill_int(int n, int* a, int v)
{
  const int t = blockIdx.x * BS + threadIdx.x;
  if (t < n) a[t] = v;
}

__global__ void k_compact_bonds(int nb, const int* keep, const int* off, const int2* ij,
                                const double4* k4, const double4* mx4, const double4* D4,
                                const int* rank, int2* ij2, double4* k42, double4* mx42,
                                double4* D42, int* rank2)
{
  const int b = blockIdx.x * BS + threadIdx.x;
  if (b >= nb || !keep[b]) return;
  const int w = off[b];
  ij2[w] = ij[b];
  k42[w] = k4[b];
  mx42[w] = mx4[b];
  D42[w] = D4[b];
  rank2[w] = rank[b];
}



// CEWallInteractionGroup::Update (EWallInteractionGroup.hpp:57-82): particles
// with |(x - o).n| < gridSpacing become candidates; isInInner (ntable.hpp:207-222)
// decides whether their force counts towards the wall force.
// The walls travel as one by-value array in the kernel arguments and are read
// in place (a local copy of the array would live in scratch memory).
struct WallSet {
  WallParam w[ESP_MAX_WALL_GROUPS];
};
__global__ void k_wall_update(PView p, GridParams g, int nwg, WallSet ws, int* mark)
{
  const int i = blockIdx.x * BS + threadIdx.x;
  unsigned fl = 0u;
  if (i < p.n) {
    fl = wall_membership(g, nwg, ws.w, p.pos[i], p.flags[i]);
    p.flags[i] = fl;
  }
  // mark[group of 64 particles]: holds wall candidates
  const unsigned long long any = __ballot(((fl >> PF_WALL_SHIFT) & 0xFFu) != 0u);
  if (mark && (threadIdx.x & 63) == 0 && i < p.n) mark[i >> 6] = any ? 1 : 0;
}

// ---------------------------------------------------------------------------
// bookkeeping of bond breaks on the device
// ---------------------------------------------------------------------------
// PIS_EB::update (pi_storage_eb.hpp:23-49) for one bond whose criterion held in
// the previous step: the bond leaves its group (marked dead, record zeroed, key
// erased from the exclusion set), both particles are flagged
// (RotBondedInteraction.cpp:211-213) and the event is logged.
__device__ __forceinline__ void break_one(PView p, const BondSet& bs, int gb, UpdState* st,
                                          int* flist, int4* evt, long long step)
{
  int g = 0;
  while (g + 1 < bs.count && gb >= bs.off[g + 1]) g++;
  const int b = gb - bs.off[g];
  if (b < 0 || b >= bs.n[g]) return;
  const int2 e = bs.ij[g][b];
  if (e.x < 0) return;
  // independent memory operations first, so their latencies overlap
  const int id1 = p.id[e.x], id2 = p.id[e.y];
  const int2 so = bs.slot_of[bs.rec_off[g] + b];
  const unsigned ox = atomicOr(&p.flags[e.x], PF_FLAG);
  const unsigned oy = atomicOr(&p.flags[e.y], PF_FLAG);
  bs.ij[g][b] = make_int2(-1, -1);
  const int ev = atomicAdd(&st->evt_count, 1);
  const int nx = (ox & PF_FLAG) ? 0 : 1, ny = (oy & PF_FLAG) ? 0 : 1;
  if (nx + ny) {
    const int f0 = atomicAdd(&st->fcount, nx + ny);
    if (nx) flist[f0] = e.x;
    if (ny) flist[f0 + nx] = e.y;
  }
  double* s0 = bs.slots + (size_t)bs.ss * so.x;
  double* s1 = bs.slots + (size_t)bs.ss * so.y;
  for (int k = 0; k < bs.ss; k++) {
    s0[k] = 0.0;
    s1[k] = 0.0;
  }
  bs.sact[so.x] = 0;
  bs.sact[so.y] = 0;
  evt[ev] = make_int4((int)step, id1, id2, 0);
  hs_erase(bs.hs[g], pair_key(id1, id2));
}

// the previous step's breaks on the host bookkeeping path
__global__ void k_break_apply(StepCtl ctl, PView p, BondSet bs, const int* broken_list,
                              UpdState* st, int* flist, int4* evt, long long step)
{
  if (step_skip(ctl)) return;
  const int nb = ctl.prev->nbroken;
  for (int t = blockIdx.x * BS + threadIdx.x; t < nb; t += gridDim.x * BS)
    break_one(p, bs, broken_list[t], st, flist, evt, step);
}

// outside the table's padded grid: erased by the next table build (the
// predicate of k_cells_count)
__device__ __forceinline__ bool outside_grid(const GridParams& g, const double4& P)
{
  int ix, iy, iz;
  return !(cell_coords(g, P.x, P.y, P.z, ix, iy, iz) && ix >= 0 && ix < g.nx && iy >= 0 &&
           iy < g.ny && iz >= 0 && iz < g.nz);
}

// k_break_apply before a table build that erases particles: the reference
// erases the particles outside the grid, with their bonds, before it tests the
// bonds (NeighborTable::build, then PIS_EB::update), so a bond with such a
// particle is left to the erasure: no break event, no flags.
__global__ void k_break_apply_erase(StepCtl ctl, PView p, BondSet bs, const int* broken_list,
                                    UpdState* st, int* flist, int4* evt, long long step,
                                    GridParams g)
{
  if (step_skip(ctl)) return;
  const int nb = ctl.prev->nbroken;
  for (int t = blockIdx.x * BS + threadIdx.x; t < nb; t += gridDim.x * BS) {
    const int gb = broken_list[t];
    int k = 0;
    while (k + 1 < bs.count && gb >= bs.off[k + 1]) k++;
    const int b = gb - bs.off[k];
    if (b < 0 || b >= bs.n[k]) continue;
    const int2 e = bs.ij[k][b];
    if (e.x >= 0 && (outside_grid(g, p.pos[e.x]) || outside_grid(g, p.pos[e.y]))) continue;
    break_one(p, bs, gb, st, flist, evt, step);
  }
}

// TSubLattice::updateInteractions after bond breaks, for a queued step, run by
// block 0 of the step's force launch while the other blocks compute the stored
// interactions: the previous step's breaks are applied (break_one), then
// getNewList (ntable.hpp:628-664) and the first dynamic group's incremental
// update (pi_storage_ed.hpp:137-156 / pi_storage_ne.hpp:79-96): pairs of
// flagged particles in neighbouring cells of the last build, without a distance
// test, minus excluded (and, for history groups, stored) pairs, are appended in
// key order and their forces of this step are computed here; then every flag
// is cleared.  The force blocks cover the appendix as it was before this step
// (n_app[1]; the gather advances it to n_app[0]).  Bonds broken in the
// previous step carry that step in D4.w, so the force blocks skip them without
// waiting for this block.  When the pairs do not fit the appendix, the queue
// halts and the host redoes the step (its input history buffer is intact).
#define NEW_SENTINEL 0x7fffffffffffffffll
template <bool RIGID>
__device__ __forceinline__ void dyn_item(const PView& p, int c, const ForceSeg& g,
                                         const ForceLaunch& fl)
{
  switch (g.kind) {
    case ESP_SEG_ROT_FRICTION: rot_friction_item<RIGID>(p, c, g, fl); break;
    case ESP_SEG_NROT_ELASTIC: nrot_elastic_item(p, c, g, fl); break;
    case ESP_SEG_ROT_ELASTIC: rot_elastic_item(p, c, g, fl); break;
    default: break;
  }
}

// RIGID, TRACK: the extended launch (rigid=True RotFriction groups; app_step,
// the pair-event log's step of each appended pair)
template <bool RIGID, bool TRACK>
__device__ void incremental_update(const StepCtl& ctl, const PView& p, const UpdParams& up,
                                   const ForceLaunch& fl, int* app_step)
{
  __shared__ long long s_key[ESP_NEW_CAP];
  __shared__ int s_cnt, s_over, s_keep;
  const int nbk = ctl.prev->nbroken;
  if (nbk <= 0) return;
  const int tid = threadIdx.x;
  for (int t = tid; t < nbk; t += BS)
    break_one(p, up.bs, up.broken_prev[t], up.st, up.flist, up.evt, up.step);
  if (!up.has_group) return;
  const DynAppend& da = up.da;
  const GridParams& g = up.g;
  // flags, flagged list and its count complete: within one workgroup a barrier
  // orders global memory (the waves share one vector L1)
  __syncthreads();
  if (tid == 0) {
    s_cnt = 0;
    s_over = 0;
    s_keep = 0;
  }
  __syncthreads();
  const int nf = up.st->fcount;
  // a cascade: four waves would take milliseconds over the flagged particles
  // while the whole chip waits, the host path takes one
  if (nf > ESP_FLAG_CAP) {
    if (tid == 0) {
      *ctl.reason = 2;
      *ctl.halted = ctl.step_id;
    }
    return;
  }
  // one wave per flagged particle; lane l scans half (l / 27) of the items of
  // neighbour cell l % 27, so the dependent loads of a cell scan run in parallel
  const int lane = tid & 63;
  for (int f = tid >> 6; f < nf; f += BS / 64) {
    const int pi = up.flist[f];
    const int c = up.cell[pi];
    const int cx = c / (g.ny * g.nz);
    const int rem = c - cx * (g.ny * g.nz);
    const int cy = rem / g.nz;
    const int cz = rem - cy * g.nz;
    const int idp = p.id[pi];
    if (lane >= 54) continue;
    const int nc = lane % 27, half = lane / 27;
    int x = cx + nc / 9 - 1;
    const int y = cy + (nc / 3) % 3 - 1, z = cz + nc % 3 - 1;
    if (g.circ_x) x = (x + g.nx) % g.nx;  // the stencil wraps in a circular x
    if (x < 0 || x >= g.nx || y < 0 || y >= g.ny || z < 0 || z >= g.nz) continue;
    const int c2 = g.ny * g.nz * x + g.nz * y + z;
    const int t0 = up.cell_start[c2], t1 = up.cell_start[c2 + 1];
    // this lane's items u = t0 + half + 2 j, four at a time with their loads in flight together
    for (int u = t0 + half; u < t1; u += 8) {
      int q[4];
      unsigned fq[4];
      int idq[4];
#pragma unroll
      for (int j = 0; j < 4; j++) q[j] = u + 2 * j < t1 ? up.cell_items[u + 2 * j] : -1;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        fq[j] = q[j] >= 0 ? p.flags[q[j]] : 0u;
        idq[j] = q[j] >= 0 ? p.id[q[j]] : 0;
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (!(fq[j] & PF_FLAG) || idq[j] <= idp) continue;
        const int k = atomicAdd(&s_cnt, 1);
        if (k < ESP_NEW_CAP) {
          s_key[k] = pair_key(pi, q[j]);
        } else {
          s_over = 1;
        }
      }
    }
  }
  __syncthreads();
  const int n = min(s_cnt, ESP_NEW_CAP);
  // keep: not excluded, not stored (history groups); others sort to the end.
  // A key holds the pair's slots (lower-id particle first).
  int m = 1;
  while (m < n) m <<= 1;
  for (int t = tid; t < m; t += BS) {
    if (t < n) {
      const long long key = s_key[t];
      const int a = (int)(key >> 32), b = (int)(key & 0xffffffffll);
      const bool keep = !rejected(da.ex, pair_key(p.id[a], p.id[b]), a, b) &&
                        !(da.is_hist && hs_find(da.present, key) >= 0);
      if (keep) atomicAdd(&s_keep, 1);
      else s_key[t] = NEW_SENTINEL;
    } else {
      s_key[t] = NEW_SENTINEL;
    }
  }
  __syncthreads();
  if (n <= BS) {
    // few candidates: each kept key moves to its rank among the kept keys (keys
    // are distinct, the sentinel is larger than any), one pass
    long long mine = NEW_SENTINEL;
    int rank = 0;
    if (tid < n) {
      mine = s_key[tid];
      if (mine != NEW_SENTINEL)
        for (int u = 0; u < n; u++) rank += s_key[u] < mine ? 1 : 0;
    }
    __syncthreads();
    if (mine != NEW_SENTINEL) s_key[rank] = mine;
    __syncthreads();
  } else {
    for (int k = 2; k <= m; k <<= 1)
      for (int j = k >> 1; j > 0; j >>= 1) {
        for (int i = tid; i < m; i += BS) {
          const int ixj = i ^ j;
          if (ixj > i) {
            const bool up_ = (i & k) == 0;
            const long long a = s_key[i], b = s_key[ixj];
            if ((a > b) == up_) {
              s_key[i] = b;
              s_key[ixj] = a;
            }
          }
        }
        __syncthreads();
      }
  }
  const int kept = s_keep;
  const int napp = da.n_app[0];
  if (napp + kept > ESP_APP_CAP) s_over = 1;
  // each new record takes the next appendix slot of both its particles, pairs
  // in key order: the slot is the count of earlier kept pairs on that particle
  for (int t = tid; t < kept; t += BS) {
    const int a = (int)(s_key[t] >> 32), b = (int)(s_key[t] & 0xffffffffll);
    int da_ = 0, db_ = 0;
    for (int u = 0; u < kept; u++) {
      const long long ku = s_key[u];
      const int a2 = (int)(ku >> 32), b2 = (int)(ku & 0xffffffffll);
      da_ += (a2 == a) | (b2 == a);
      db_ += (a2 == b) | (b2 == b);
    }
    if (up.xcnt[a] + da_ > ESP_XSLOTS || up.xcnt[b] + db_ > ESP_XSLOTS) s_over = 1;
  }
  __syncthreads();
  if (s_over) {
    if (tid == 0) {
      *ctl.reason = 2;
      *ctl.halted = ctl.step_id;
    }
    return;
  }
  for (int t = tid; t < kept; t += BS) {
    const long long key = s_key[t];
    const int a = (int)(key >> 32), b = (int)(key & 0xffffffffll);
    int pa = 0, pb = 0;
    for (int u = 0; u < t; u++) {
      const long long ku = s_key[u];
      const int a2 = (int)(ku >> 32), b2 = (int)(ku & 0xffffffffll);
      pa += (a2 == a) | (b2 == a);
      pb += (a2 == b) | (b2 == b);
    }
    const int w = da.n_main + napp + t;
    da.ij[w] = make_int2(a, b);
    da.key[w] = key;
    if (da.ff) da.ff[w] = make_double4(0.0, 0.0, 0.0, 0.0);
    if (TRACK && app_step) app_step[napp + t] = (int)up.step;
    if (da.is_hist) hs_insert(da.present, key);
    // appendix slots start at zero (cleared at the last rebuild, used once)
    da.slot_of[da.app_rec_off + napp + t] =
        make_int2(da.xbase + ESP_XSLOTS * a + up.xcnt[a] + pa, da.xbase + ESP_XSLOTS * b + up.xcnt[b] + pb);
  }
  __syncthreads();  // every xcnt read above precedes the increments
  for (int t = tid; t < kept; t += BS) {
    const long long key = s_key[t];
    atomicAdd(&up.xcnt[(int)(key >> 32)], 1);
    atomicAdd(&up.xcnt[(int)(key & 0xffffffffll)], 1);
  }
  // this step's forces of the new pairs (each entry was written by the same thread)
  const ForceSeg& us = fl.seg[up.useg];
  const int c0 = da.n_main + napp;
  for (int t = tid; t < kept; t += BS) dyn_item<RIGID>(p, c0 + t, us, fl);
  if (tid == 0) da.n_app[0] = napp + kept;
  for (int t = tid; t < nf; t += BS) p.flags[up.flist[t]] &= ~PF_FLAG;
  if (tid == 0) up.st->fcount = 0;
}

// The force laws of every interaction group in one launch: each segment of
// blocks covers one group (bonded groups first, their law is the longest), so
// the groups' memory latencies overlap.  Every interaction writes its slots.
// In a queued step block 0 runs the incremental update (fl.ublk).
template <bool RIGID, bool TRACK>
__device__ __forceinline__ void forces_body(const StepCtl& ctl, const PView& p,
                                            const ForceLaunch& fl, const UpdParams& up,
                                            int* app_step)
{
  if (step_skip(ctl)) return;
  if (fl.ublk && blockIdx.x == 0) {
    incremental_update<RIGID, TRACK>(ctl, p, up, fl, app_step);
    return;
  }
  const int vb = (int)blockIdx.x - fl.ublk;
  int s = 0;
  while (s + 1 < fl.count && vb >= fl.seg[s + 1].blk0) s++;
  const ForceSeg& g = fl.seg[s];
  // blocks go round-robin to the 8 XCDs: within a segment each XCD takes a
  // contiguous range of blocks, so the state of particles shared by
  // neighbouring interactions is fetched into one L2 (a bijection on the
  // segment's blocks)
  const int nseg = (s + 1 < fl.count ? fl.seg[s + 1].blk0 : fl.nblocks) - g.blk0;
  const int b0 = g.blk0 + fl.ublk;  // launch index of the segment's first block
  const int d = ((int)blockIdx.x - b0) & 7;
  const int q8 = nseg >> 3, r8 = nseg & 7;
  const int lbk = d * q8 + min(d, r8) + ((int)blockIdx.x - b0 - d) / 8;
  const int c = lbk * BS + (int)threadIdx.x;
  if (g.kind == ESP_SEG_ROT_BOND) {
    rot_bond_item(ctl, p, c, g, fl);
  } else if (c < g.n + *g.n_app) {
    dyn_item<RIGID>(p, c, g, fl);
  }
}

__global__ __launch_bounds__(BS, 4) void k_forces(StepCtl ctl, PView p, ForceLaunch fl, UpdParams up)
{
  if (step_skip(ctl)) return;
  if (fl.ublk && blockIdx.x == 0) {
    incremental_update<false, false>(ctl, p, up, fl, nullptr);
    return;
  }
  const int vb = (int)blockIdx.x - fl.ublk;
  int s = 0;
  while (s + 1 < fl.count && vb >= fl.seg[s + 1].blk0) s++;
  const ForceSeg& g = fl.seg[s];
  // blocks go round-robin to the 8 XCDs: within a segment each XCD takes a
  // contiguous range of blocks, so the state of particles shared by
  // neighbouring interactions is fetched into one L2 (a bijection on the
  // segment's blocks)
  const int nseg = (s + 1 < fl.count ? fl.seg[s + 1].blk0 : fl.nblocks) - g.blk0;
  const int b0 = g.blk0 + fl.ublk;  // launch index of the segment's first block
  const int d = ((int)blockIdx.x - b0) & 7;
  const int q8 = nseg >> 3, r8 = nseg & 7;
  const int lbk = d * q8 + min(d, r8) + ((int)blockIdx.x - b0 - d) / 8;
  const int c = lbk * BS + (int)threadIdx.x;
  if (g.kind == ESP_SEG_ROT_BOND) {
    rot_bond_item(ctl, p, c, g, fl);
  } else if (c < g.n + *g.n_app) {
    dyn_item<false>(p, c, g, fl);
  }
}

// the same launch with a rigid=True RotFriction group or a tracked group (the
// rigid law needs more registers than the common kernel's budget of 128, so
// this kernel has no minimum occupancy: it runs without register spills)
__global__ __launch_bounds__(BS) void k_forces_ext(StepCtl ctl, PView p, ForceLaunch fl,
                                                      UpdParams up, ForceExt ext)
{
  forces_body<true, true>(ctl, p, fl, up, ext.app_step);
}

__global__ void k_hash_clear(HashRef h)
{
  const unsigned t = blockIdx.x * BS + threadIdx.x;
  if (t <= h.mask) h.t[t] = HS_EMPTY;
}

__global__ void k_hash_insert(HashRef h, const long long* keys, int n)
{
  const int t = blockIdx.x * BS + threadIdx.x;
  if (t < n) hs_insert(h, keys[t]);
}

__global__ void k_bond_keys(int nb, const int2* ij, const int* id, long long* keys)
{
  const int b = blockIdx.x * BS + threadIdx.x;
  if (b >= nb) return;
  const int2 e = ij[b];
  keys[b] = e.x < 0 ? -1ll : pair_key(id[e.x], id[e.y]);
}

__global__ void k_alive_flags(int nb, const int2* ij, int* keep)
{
  const int b = blockIdx.x * BS + threadIdx.x;
  if (b < nb) keep[b] = ij[b].x >= 0 ? 1 : 0;
}

// ---------------------------------------------------------------------------
// per-particle CSR of force records
// ---------------------------------------------------------------------------
__global__ void k_inc_count(int nc, const int2* ij, int* cnt)
{
  const int c = blockIdx.x * BS + threadIdx.x;
  if (c >= nc) return;
  const int2 e = ij[c];
  if (e.x < 0) return;
  atomicAdd(&cnt[e.x], 1);
  atomicAdd(&cnt[e.y], 1);
}

// CSR entry of an interaction for each of its particles: the record reference
// (rec << 2 | has-moments << 1 | second-particle) in the low 32 bits, above it
// the summation order: group position (5 bits) and the interaction's rank in
// the group's reference order (27 bits; the storage index where storage order
// is that order).
__global__ void k_inc_fill(int nc, const int2* ij, int rec_off, int has_m, const int* rank,
                           unsigned long long grp, const int* off, int* fill,
                           unsigned long long* ent)
{
  const int c = blockIdx.x * BS + threadIdx.x;
  if (c >= nc) return;
  const int2 e = ij[c];
  if (e.x < 0) return;
  const unsigned v = ((unsigned)(rec_off + c) << 2) | ((unsigned)has_m << 1);
  const unsigned long long hi = (grp << 59) | ((unsigned long long)(rank ? rank[c] : c) << 32);
  ent[off[e.x] + atomicAdd(&fill[e.x], 1)] = hi | v;
  ent[off[e.y] + atomicAdd(&fill[e.y], 1)] = hi | v | 1u;
}

// Each interaction's place in its two particles' runs, in summation order: the
// number of smaller entries of the run (the runs are short and shared by
// neighbouring threads, so the reads stay in L1; sorting a run in one thread took
// 0.8 ms where flagged pairs made runs of 200).  slot_of[record] = the two places;
// with ent given, the places are filled instead: ent[place] = (the other
// particle, bit 31: this one is the second; record).
__global__ void k_inc_rank(int nc, const int2* ij, int rec_off, int has_m, const int* rank,
                           unsigned long long grp, const int* off, const unsigned long long* ent64,
                           int2* slot_of, int2* ent)
{
  const int t = blockIdx.x * BS + threadIdx.x;
  const int c = t >> 1, side = t & 1;
  if (c >= nc) return;
  const int2 e = ij[c];
  if (e.x < 0) return;
  const unsigned v = ((unsigned)(rec_off + c) << 2) | ((unsigned)has_m << 1) | (unsigned)side;
  const unsigned long long mine =
      (grp << 59) | ((unsigned long long)(rank ? rank[c] : c) << 32) | v;
  const int p = side ? e.y : e.x;
  const int a = off[p], b = off[p + 1];
  int r = a;
  for (int k = a; k < b; k++) r += ent64[k] < mine ? 1 : 0;
  if (ent)
    ent[r] = make_int2(side ? (e.x | (int)0x80000000u) : e.y, rec_off + c);
  else
    reinterpret_cast<int*>(slot_of + rec_off + c)[side] = r;
}

// ---------------------------------------------------------------------------
// exclusive scan (1024 elements per block, recursive over block sums)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(BS) void k_scan_local(const int* in, int nvalid, int* out, int m, int* bsum)
{
  __shared__ int s[BS];
  const int base = blockIdx.x * 4 * BS + threadIdx.x * 4;
  int v[4];
  int acc = 0;
  for (int k = 0; k < 4; k++) {
    const int idx = base + k;
    v[k] = (idx < nvalid) ? in[idx] : 0;
    acc += v[k];
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int o = 1; o < BS; o <<= 1) {
    const int t = threadIdx.x >= o ? s[threadIdx.x - o] : 0;
    __syncthreads();
    s[threadIdx.x] += t;
    __syncthreads();
  }
  int run = s[threadIdx.x] - acc;  // exclusive prefix of this thread
  for (int k = 0; k < 4; k++) {
    const int idx = base + k;
    if (idx < m) out[idx] = run;
    run += v[k];
  }
  if (bsum && threadIdx.x == BS - 1) bsum[blockIdx.x] = s[BS - 1];
}

// Short arrays in one block and one launch: V values a thread, all loaded at
// once, the sums of a wave by shuffles, the waves' through LDS.  A thread's values
// are consecutive, so every load of a wave touches 64 lines: bound by the line
// look-ups of one CU, which 16-byte loads and stores (`vec`: both arrays are so
// aligned) cut to a quarter.  15,000 values 16.3 -> 4.0 us.
#define SCAN_ONE 32768
template <int V>
__global__ __launch_bounds__(1024) void k_scan_one(const int* in, int nvalid, int* out, int m,
                                                   int vec)
{
  __shared__ int wsum[16];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int base = t * V;
  int v[V], acc = 0;
  if (vec && base + V <= nvalid) {
#pragma unroll
    for (int k = 0; k < V; k += 4) {
      const int4 q = *reinterpret_cast<const int4*>(in + base + k);
      v[k] = q.x; v[k + 1] = q.y; v[k + 2] = q.z; v[k + 3] = q.w;
    }
  } else {
#pragma unroll
    for (int k = 0; k < V; k++) v[k] = base + k < nvalid ? in[base + k] : 0;
  }
#pragma unroll
  for (int k = 0; k < V; k++) acc += v[k];
  int inc = acc;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(inc, d, 64);
    if (lane >= d) inc += u;
  }
  if (lane == 63) wsum[wv] = inc;
  __syncthreads();
  int run = inc - acc;
#pragma unroll
  for (int w = 0; w < 16; w++) run += w < wv ? wsum[w] : 0;
  if (vec && base + V <= m) {
#pragma unroll
    for (int k = 0; k < V; k += 4) {
      int4 q;
      q.x = run; run += v[k];
      q.y = run; run += v[k + 1];
      q.z = run; run += v[k + 2];
      q.w = run; run += v[k + 3];
      *reinterpret_cast<int4*>(out + base + k) = q;
    }
  } else {
#pragma unroll
    for (int k = 0; k < V; k++) {
      if (base + k < m) out[base + k] = run;
      run += v[k];
    }
  }
}

__global__ void k_scan_add(int* out, int m, const int* boff)
{
  const int idx = blockIdx.x * 4 * BS + threadIdx.x * 4;
  const int add = boff[blockIdx.x];
  for (int k = 0; k < 4; k++)
    if (idx + k < m) out[idx + k] += add;
}

static size_t scan_tmp_rec(long long m)
{
  const long long nb = (m + 4 * BS - 1) / (4 * BS);
  if (nb <= 1) return 0;
  return (size_t)(2 * nb) + scan_tmp_rec(nb);
}

size_t scan_tmp_size(int n) { return scan_tmp_rec((long long)n + 1) + 16; }

static void scan_rec(hipStream_t s, const int* in, int nvalid, int* out, int m, int* tmp)
{
  if (m <= SCAN_ONE) {
    const int vec = (((uintptr_t)in | (uintptr_t)out) & 15) == 0;
    const auto scan = m <= SCAN_ONE / 4   ? k_scan_one<8>
                      : m <= SCAN_ONE / 2 ? k_scan_one<16>
                                          : k_scan_one<32>;
    hipLaunchKernelGGL(scan, dim3(1), dim3(1024), 0, s, in, nvalid, out, m, vec);
    return;
  }
  const int nb = (m + 4 * BS - 1) / (4 * BS);
  int* bsum = nb > 1 ? tmp : nullptr;
  hipLaunchKernelGGL(k_scan_local, dim3(nb), dim3(BS), 0, s, in, nvalid, out, m, bsum);
  if (nb > 1) {
    int* boff = tmp + nb;
    scan_rec(s, bsum, nb, boff, nb, tmp + 2 * nb);
    hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(BS), 0, s, out, m, boff);
  }
}

void launch_exclusive_scan(hipStream_t s, const int* in, int* out, int n, int* tmp)
{
  scan_rec(s, in, n, out, n + 1, tmp);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
int gather_blocks(int n) { return n > 0 ? nblk(n) : 0; }

int force_blocks(int n) { return nblk(n); }

// With a pair of events (ev_a, ev_b both set) the launch stamps them itself at
// the kernel's start and end (hipExtLaunchKernelGGL), so their elapsed time is
// the kernel's own execution time; false when nothing was launched.
bool launch_forces(hipStream_t s, StepCtl ctl, PView p, const ForceLaunch& fl,
                   const UpdParams* up, hipEvent_t ev_a, hipEvent_t ev_b, const ForceExt* ext)
{
  UpdParams u;
  if (up) {
    u = *up;
  } else {
    memset(&u, 0, sizeof u);
  }
  ForceLaunch f = fl;
  f.ublk = up ? 1 : 0;
  if (f.nblocks + f.ublk <= 0) return false;
  bool extended = ext && ext->app_step;
  for (int k = 0; k < f.count; k++)
    extended |= f.seg[k].kind == ESP_SEG_ROT_FRICTION && f.seg[k].rigid;
  ForceExt x;
  memset(&x, 0, sizeof x);
  if (ext) x = *ext;
  if (ev_a && ev_b) {
    if (extended)
      hipExtLaunchKernelGGL(k_forces_ext, dim3(f.nblocks + f.ublk), dim3(BS), 0, s, ev_a, ev_b, 0,
                            ctl, p, f, u, x);
    else
      hipExtLaunchKernelGGL(k_forces, dim3(f.nblocks + f.ublk), dim3(BS), 0, s, ev_a, ev_b, 0, ctl,
                            p, f, u);
  } else if (extended) {
    hipLaunchKernelGGL(k_forces_ext, dim3(f.nblocks + f.ublk), dim3(BS), 0, s, ctl, p, f, u, x);
  } else {
    hipLaunchKernelGGL(k_forces, dim3(f.nblocks + f.ublk), dim3(BS), 0, s, ctl, p, f, u);
  }
  return true;
}

void launch_break_apply(hipStream_t s, StepCtl ctl, PView p, BondSet bs, const int* broken_list,
                        UpdState* st, int* flist, int4* evt, long long step,
                        const GridParams* erase_grid)
{
  if (bs.count <= 0) return;
  if (erase_grid)
    hipLaunchKernelGGL(k_break_apply_erase, dim3(16), dim3(BS), 0, s, ctl, p, bs, broken_list, st,
                       flist, evt, step, *erase_grid);
  else
    hipLaunchKernelGGL(k_break_apply, dim3(16), dim3(BS), 0, s, ctl, p, bs, broken_list, st, flist,
                       evt, step);
}

void launch_hash_clear(hipStream_t s, HashRef h)
{
  hipLaunchKernelGGL(k_hash_clear, dim3(nblk((long long)h.mask + 1)), dim3(BS), 0, s, h);
}

void launch_hash_insert(hipStream_t s, HashRef h, const long long* keys, int n)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_hash_insert, dim3(nblk(n)), dim3(BS), 0, s, h, keys, n);
}

void launch_bond_keys(hipStream_t s, int nb, const int2* ij, const int* id, long long* keys)
{
  if (nb <= 0) return;
  hipLaunchKernelGGL(k_bond_keys, dim3(nblk(nb)), dim3(BS), 0, s, nb, ij, id, keys);
}

void launch_alive_flags(hipStream_t s, int nb, const int2* ij, int* keep)
{
  if (nb <= 0) return;
  hipLaunchKernelGGL(k_alive_flags, dim3(nblk(nb)), dim3(BS), 0, s, nb, ij, keep);
}

static bool extra_forces(const GatherParams& gp)
{
  bool extra = gp.ndamp > 0;
  for (int w = 0; w < gp.nwg; w++) extra |= gp.wall[w].bonded != 0 || gp.wall[w].tagged != 0;
  return extra;
}

template <class K>
static void gather_launch(K kern, int blocks, hipStream_t s, StepCtl ctl, PView p,
                          const GatherParams& gp, hipEvent_t ev_a, hipEvent_t ev_b)
{
  if (ev_a && ev_b)
    hipExtLaunchKernelGGL(kern, dim3(blocks), dim3(BS), 0, s, ev_a, ev_b, 0, ctl, p, gp);
  else
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(BS), 0, s, ctl, p, gp);
}

// above this many particles one lane a particle: both forms take the same time
// at 100,000 (15.9 and 15.4 us); at 64,000 particles one lane each is one wave
// for every SIMD of the chip
#define GATHER_WIDE 65536
// three active slots a lane in flight up to this many, see k_gather_integrate
#define GATHER_DEEP 32768
bool launch_gather_integrate(hipStream_t s, StepCtl ctl, PView p, const GatherParams& gp,
                             hipEvent_t ev_a, hipEvent_t ev_b)
{
  if (p.n <= 0) return false;
  const bool extra = extra_forces(gp);
  if (gp.sig) {
    if (extra) gather_launch(k_gather_stress<true>, nblk(p.n), s, ctl, p, gp, ev_a, ev_b);
    else gather_launch(k_gather_stress<false>, nblk(p.n), s, ctl, p, gp, ev_a, ev_b);
  } else if (p.n > GATHER_WIDE) {
    if (extra) gather_launch(k_gather_wide<true>, nblk(p.n), s, ctl, p, gp, ev_a, ev_b);
    else gather_launch(k_gather_wide<false>, nblk(p.n), s, ctl, p, gp, ev_a, ev_b);
  } else {
    const auto deep = extra ? k_gather_integrate<true, 3> : k_gather_integrate<false, 3>;
    const auto flat = extra ? k_gather_integrate<true, 1> : k_gather_integrate<false, 1>;
    gather_launch(p.n <= GATHER_DEEP ? deep : flat, nblk(p.n, 64), s, ctl, p, gp, ev_a, ev_b);
  }
  return true;
}

// BrittleBeamSCInteraction::broken for every live bond of the stress-criterion
// groups, on the positions after this step's integration and the stresses of
// its forces - the state the reference's next updateInteractions sees.
__global__ __launch_bounds__(BS) void k_sc_break(StepCtl ctl, PView p, ScLaunch sl)
{
  if (step_skip(ctl)) return;
  int g = 0;
  while (g + 1 < sl.count && (int)blockIdx.x >= sl.blk0[g + 1]) g++;
  const int b = ((int)blockIdx.x - sl.blk0[g]) * BS + (int)threadIdx.x;
  if (b >= sl.n[g]) return;
  const int2 e = sl.ij[g][b];
  if (e.x < 0) return;
  const double4 P1 = p.pos[e.x], P2 = x_image(P1, p.pos[e.y], sl.period);
  if (esp_sc_broken(xyz(P1), P1.w, sl.sig + 9 * (size_t)e.x, xyz(P2), P2.w,
                    sl.sig + 9 * (size_t)e.y, sl.sigma3[g], sl.cohesion[g], sl.tan_angle[g])) {
    sl.D4[g][b].w = sl.step;
    const int slot = atomicAdd(&ctl.cur->nbroken, 1);
    sl.broken_list[slot] = sl.bond_off[g] + b;
  }
}

void launch_sc_break(hipStream_t s, StepCtl ctl, PView p, const ScLaunch& sl)
{
  if (sl.nblocks <= 0) return;
  hipLaunchKernelGGL(k_sc_break, dim3(sl.nblocks), dim3(BS), 0, s, ctl, p, sl);
}

void launch_batch_end(hipStream_t s, const BatchEnd& be)
{
  const dim3 g(be.nwg > 0 ? be.nsteps : 1), b(BS);
  if (be.list)
    hipLaunchKernelGGL((k_batch_end<true>), g, b, 0, s, be);
  else
    hipLaunchKernelGGL((k_batch_end<false>), g, b, 0, s, be);
}

template <class K>
static void contact_launch(K kern, dim3 g, hipStream_t s, StepCtl ctl, PView p,
                           const ContactLaunch& cl, const GatherParams& gp, hipEvent_t ev_a,
                           hipEvent_t ev_b)
{
  if (ev_a && ev_b)
    hipExtLaunchKernelGGL(kern, g, dim3(BS), 0, s, ev_a, ev_b, 0, ctl, p, cl, gp);
  else
    hipLaunchKernelGGL(kern, g, dim3(BS), 0, s, ctl, p, cl, gp);
}

int contact_groups(int n) { return nblk(n, 64); }

bool launch_contact_step(hipStream_t s, StepCtl ctl, PView p, const ContactLaunch& cl,
                         const GatherParams& gp, hipEvent_t ev_a, hipEvent_t ev_b)
{
  if (p.n <= 0) return false;
  const bool extra = extra_forces(gp);
  if (cl.count == 1 && cl.seg[0].kind == ESP_SEG_NROT_ELASTIC) {
    constexpr int G = 4;  // lanes a particle: its 7 or so pairs in two rounds
    const dim3 g(nblk(p.n, BS / G));
    if (extra) contact_launch(k_contact_step<true, G>, g, s, ctl, p, cl, gp, ev_a, ev_b);
    else contact_launch(k_contact_step<false, G>, g, s, ctl, p, cl, gp, ev_a, ev_b);
    return true;
  }
  const dim3 g(nblk(p.n, 64));
  if (cl.count == 1 && cl.seg[0].kind == ESP_SEG_ROT_FRICTION && !cl.seg[0].rigid) {
    if (extra) contact_launch(k_contact_block<true, ESP_SEG_ROT_FRICTION>, g, s, ctl, p, cl, gp, ev_a, ev_b);
    else contact_launch(k_contact_block<false, ESP_SEG_ROT_FRICTION>, g, s, ctl, p, cl, gp, ev_a, ev_b);
  } else {
    if (extra) contact_launch(k_contact_block<true, 0>, g, s, ctl, p, cl, gp, ev_a, ev_b);
    else contact_launch(k_contact_block<false, 0>, g, s, ctl, p, cl, gp, ev_a, ev_b);
  }
  return true;
}

void launch_wall_list(hipStream_t s, int ng, const int* mark, int* list, int* list_n)
{
  hipLaunchKernelGGL(k_wall_list, dim3(1), dim3(1024), 0, s, ng, mark, list, list_n);
}

void launch_cells_count(hipStream_t s, PView p, GridParams g, int* cell, int* cell_count,
                        int* n_out)
{
  if (p.n <= 0) return;
  hipLaunchKernelGGL(k_cells_count, dim3(nblk(p.n)), dim3(BS), 0, s, p, g, cell, cell_count, n_out);
}

void launch_cells_fill(hipStream_t s, int n, const int* cell, const int* cell_start,
                       int* cell_fill, int* cell_items)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_cells_fill, dim3(nblk(n)), dim3(BS), 0, s, n, cell, cell_start, cell_fill,
                     cell_items);
}

void launch_cells_sort(hipStream_t s, int ncell, const int* cell_start, int* cell_items)
{
  if (ncell <= 0) return;
  hipLaunchKernelGGL(k_cells_sort, dim3(nblk(ncell)), dim3(BS), 0, s, ncell, cell_start, cell_items);
}

void launch_pairs(hipStream_t s, int mode_emit, int flagged, PView p, GridParams g, double alpha,
                  const int* cell, const int* cell_start, const int* cell_items, int* cnt,
                  const int* off, int cap, int* out_p, int* out_q, long long* out_key)
{
  if (p.n <= 0) return;
  const dim3 gr(nblk(p.n, BS / 32)), bl(BS);
#define ESP_PAIRS(E, F)                                                                         \
  hipLaunchKernelGGL((k_pairs<E, F>), gr, bl, 0, s, p, g, alpha, cell, cell_start, cell_items, \
                     cnt, off, cap, out_p, out_q, out_key)
  if (mode_emit) {
    if (flagged) ESP_PAIRS(true, true);
    else ESP_PAIRS(true, false);
  } else {
    if (flagged) ESP_PAIRS(false, true);
    else ESP_PAIRS(false, false);
  }
#undef ESP_PAIRS
}

void launch_keep_cells(hipStream_t s, int n, const int* cell, int* keep)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_keep_cells, dim3(nblk(n)), dim3(BS), 0, s, n, cell, keep);
}

void launch_new_slot(hipStream_t s, int n, const int* keep, const int* off, int* nslot)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_new_slot, dim3(nblk(n)), dim3(BS), 0, s, n, keep, off, nslot);
}

template <class T>
static void compact_field(hipStream_t s, int n, int width, const int* keep, const int* off,
                          const T* src, T* dst)
{
  if (n <= 0) return;
  hipLaunchKernelGGL((k_compact_field<T>), dim3(nblk(n)), dim3(BS), 0, s, n, width, keep, off, src,
                     dst);
}
void launch_compact_field(hipStream_t s, int n, int width, const int* keep, const int* off,
                          const double4* src, double4* dst)
{
  compact_field(s, n, width, keep, off, src, dst);
}
void launch_compact_field(hipStream_t s, int n, int width, const int* keep, const int* off,
                          const double* src, double* dst)
{
  compact_field(s, n, width, keep, off, src, dst);
}
void launch_compact_field(hipStream_t s, int n, int width, const int* keep, const int* off,
                          const int* src, int* dst)
{
  compact_field(s, n, width, keep, off, src, dst);
}
void launch_compact_field(hipStream_t s, int n, int width, const int* keep, const int* off,
                          const unsigned* src, unsigned* dst)
{
  compact_field(s, n, width, keep, off, src, dst);
}

void launch_remap_pairs(hipStream_t s, int nc, const int2* ij, const int* nslot, int2* out,
                        int* keep)
{
  if (nc <= 0) return;
  hipLaunchKernelGGL(k_remap_pairs, dim3(nblk(nc)), dim3(BS), 0, s, nc, ij, nslot, out, keep);
}

void launch_pack_dyn(hipStream_t s, int nc, const int* keep, const int* off, const int2* ij,
                     const double4* ff, int2* oij, long long* okey, double4* off_)
{
  if (nc <= 0) return;
  hipLaunchKernelGGL(k_pack_dyn, dim3(nblk(nc)), dim3(BS), 0, s, nc, keep, off, ij, ff, oij, okey,
                     off_);
}

void launch_wall_cands(hipStream_t s, PView p, int w, const double4* init, int cap, int* cnt,
                       int* slot, unsigned* flg, double4* pos, double4* ipos)
{
  if (p.n <= 0) return;
  hipLaunchKernelGGL(k_wall_cands, dim3(nblk(p.n)), dim3(BS), 0, s, p, w, init, cap, cnt, slot,
                     flg, pos, ipos);
}

void launch_wall_mark_ordered(hipStream_t s, int no, const int* ord_slot, const unsigned* flags,
                              int w, int* mark)
{
  if (no <= 0) return;
  hipLaunchKernelGGL(k_wall_mark_ordered, dim3(nblk(no)), dim3(BS), 0, s, no, ord_slot, flags, w,
                     mark);
}

void launch_servo_sums(hipStream_t s, PView p, const WallParam& W, int w, int do2d,
                       const double4* init, const int* list, const int* list_n, double* out)
{
  hipLaunchKernelGGL(k_servo_sums, dim3(ESP_SERVO_BLOCKS), dim3(BS), 0, s, p, W, w, do2d,
                     contact_groups(p.n), init, list, list_n, out);
}

void launch_pack_ordered(hipStream_t s, int n, const int* order, const double4* src, int width,
                         double* out)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_pack_ordered, dim3(nblk(n)), dim3(BS), 0, s, n, order, src, width, out);
}

void launch_wall_pack_ordered(hipStream_t s, int no, const int* ord_slot, const int* mark,
                              const int* off, PView p, const double4* init, WallCand* out)
{
  if (no <= 0) return;
  hipLaunchKernelGGL(k_wall_pack_ordered, dim3(nblk(no)), dim3(BS), 0, s, no, ord_slot, mark, off,
                     p, init, out);
}

__global__ void k_report3(const int* a, const int* b, const int* c, int* out)
{
  if (threadIdx.x < 3) out[threadIdx.x] = *(threadIdx.x == 0 ? a : threadIdx.x == 1 ? b : c);
}

void launch_report3(hipStream_t s, const int* a, const int* b, const int* c, int* out)
{
  hipLaunchKernelGGL(k_report3, dim3(1), dim3(64), 0, s, a, b, c, out);
}

// several arrays to zero in one launch
__global__ void k_clear(ClearSet c)
{
  for (int k = 0; k < c.count; k++)
    for (int i = blockIdx.x * BS + threadIdx.x; i < c.n[k]; i += gridDim.x * BS) c.p[k][i] = 0;
}

void launch_clear(hipStream_t s, const ClearSet& c)
{
  int most = 0;
  for (int k = 0; k < c.count; k++) most = max(most, c.n[k]);
  if (most > 0) hipLaunchKernelGGL(k_clear, dim3(min(nblk(most), 1024)), dim3(BS), 0, s, c);
}

void launch_fill_int(hipStream_t s, int n, int* a, int v)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill_int, dim3(nblk(n)), dim3(BS), 0, s, n, a, v);
}

void launch_clear_flag_bit(hipStream_t s, PView p, UpdState* st)
{
  hipLaunchKernelGGL(k_clear_flag_bit, dim3(nblk(p.n > 0 ? p.n : 1)), dim3(BS), 0, s, p, st);
}

void launch_ed_mark(hipStream_t s, int nc, const int* cp, const int* cq, const long long* ckey,
                    ExclSet ex, const long long* okey, int nold, const int2* oij, PView p,
                    double period, int* keep, int* src, const int* nc_dev)
{
  if (nc <= 0) return;
  hipLaunchKernelGGL(k_ed_mark, dim3(nblk(nc)), dim3(BS), 0, s, nc, nc_dev, cp, cq, ckey, ex, okey, nold,
                     oij, p, period, keep, src);
}

__global__ void k_wrap_x(PView p, double x0, double period, double4* init)
{
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i >= p.n) return;
  double4 P = p.pos[i];
  double sh = 0.0;
  if (P.x < x0) sh = period;
  else if (P.x >= x0 + period) sh = -period;
  if (sh == 0.0) return;
  P.x = P.x + sh;
  p.pos[i] = P;
  double4 O = p.old[i];
  O.x = O.x + sh;
  p.old[i] = O;
  if (init) {
    double4 I = init[i];
    I.x = I.x + sh;
    init[i] = I;
  }
}

void launch_wrap_x(hipStream_t s, PView p, double x0, double period, double4* init)
{
  if (p.n <= 0) return;
  hipLaunchKernelGGL(k_wrap_x, dim3(nblk(p.n)), dim3(BS), 0, s, p, x0, period, init);
}

void launch_ne_mark(hipStream_t s, int nc, const int* cp, const int* cq, const int* id, ExclSet ex,
                    int* keep, const int* nc_dev)
{
  if (nc <= 0) return;
  hipLaunchKernelGGL(k_ne_mark, dim3(nblk(nc)), dim3(BS), 0, s, nc, nc_dev, cp, cq, id, ex, keep);
}

void launch_pair_emit(hipStream_t s, int nc, const int* keep, const int* off, const int* cp,
                      const int* cq, const long long* ckey, const int* src, const double4* off_ff,
                      int cap, int2* nij, long long* nkey, double4* nff)
{
  if (nc <= 0) return;
  hipLaunchKernelGGL(k_pair_emit, dim3(nblk(nc)), dim3(BS), 0, s, nc, keep, off, cp, cq, ckey, src,
                     off_ff, cap, nij, nkey, nff);
}

void launch_filter_new(hipStream_t s, int nc, const int* cp, const int* cq, const int* id,
                       const long long* ckey, ExclSet ex, HashRef present, int check_present,
                       int* keep)
{
  if (nc <= 0) return;
  hipLaunchKernelGGL(k_filter_new, dim3(nblk(nc)), dim3(BS), 0, s, nc, cp, cq, id, ckey, ex,
                     present, check_present, keep);
}

void launch_merge(hipStream_t s, int nold, const int2* oij, const long long* okey,
                  const double4* off_, int nnew, const int2* nij_in, const long long* nkey_in,
                  const double4* nff_in, int2* ij_out, long long* key_out, double4* ff_out)
{
  if (nold + nnew <= 0) return;
  hipLaunchKernelGGL(k_merge, dim3(nblk((long long)nold + nnew)), dim3(BS), 0, s, nold, oij, okey,
                     off_, nnew, nij_in, nkey_in, nff_in, ij_out, key_out, ff_out);
}

void launch_pack_pairs(hipStream_t s, int n, const int* keep, const int* off, const int* cp,
                       const int* cq, const long long* ckey, int2* ij, long long* key)
{
  if (n <= 0) return;
  hipLaunchKernelGGL(k_pack_pairs, dim3(nblk(n)), dim3(BS), 0, s, n, keep, off, cp, cq, ckey, ij, key);
}


void launch_compact_bonds(hipStream_t s, int nb, const int* keep, const int* off,
                          const int2* ij, const double4* k4, const double4* mx4,
                          const double4* D4, const int* rank, int2* ij2, double4* k42,
                          double4* mx42, double4* D42, int* rank2)
{
  if (nb <= 0) return;
  hipLaunchKernelGGL(k_compact_bonds, dim3(nblk(nb)), dim3(BS), 0, s, nb, keep, off, ij, k4, mx4,
                     D4, rank, ij2, k42, mx42, D42, rank2);
}



void launch_wall_update(hipStream_t s, PView p, GridParams g, int nwg, const WallParam* w, int* mark)
{
  if (p.n <= 0) return;
  WallSet ws;
  for (int k = 0; k < ESP_MAX_WALL_GROUPS; k++) ws.w[k] = w[k];
  hipLaunchKernelGGL(k_wall_update, dim3(nblk(p.n)), dim3(BS), 0, s, p, g, nwg, ws, mark);
}

void launch_inc_count(hipStream_t s, int nc, const int2* ij, int* inc_cnt)
{
  if (nc <= 0) return;
  hipLaunchKernelGGL(k_inc_count, dim3(nblk(nc)), dim3(BS), 0, s, nc, ij, inc_cnt);
}

void launch_inc_fill(hipStream_t s, int nc, const int2* ij, int rec_off, int has_m, const int* rank,
                     int grp, const int* inc_off, int* inc_fill, unsigned long long* ent64)
{
  if (nc <= 0) return;
  hipLaunchKernelGGL(k_inc_fill, dim3(nblk(nc)), dim3(BS), 0, s, nc, ij, rec_off, has_m, rank,
                     (unsigned long long)grp, inc_off, inc_fill, ent64);
}

void launch_inc_rank(hipStream_t s, int nc, const int2* ij, int rec_off, int has_m, const int* rank,
                     int grp, const int* inc_off, const unsigned long long* ent64, int2* slot_of,
                     int2* ent)
{
  if (nc <= 0) return;
  hipLaunchKernelGGL(k_inc_rank, dim3(nblk(2ll * nc)), dim3(BS), 0, s, nc, ij, rec_off, has_m, rank,
                     (unsigned long long)grp, inc_off, ent64, slot_of, ent);
}
